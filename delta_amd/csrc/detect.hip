// detect.hip — particle-pair narrow phase: the reference's drivers bf,
// penalty, hybridWithPer{Batch,Triangle}FallBack, penaltyStat and
// hybrid{Batch,Triangle}Stat (bf.cpp:28-149, penalty.cpp:50-241,
// hybrid.cpp:59-627) over a batch of particle pairs.
//
// A particle pair's rows (triangles of A) are split into `tiles` contiguous
// ranges, one workgroup (4 waves) per range, which walks its rows' triangle
// pairs in row-major chunks of 256.  Several workgroups per particle pair
// keep the CUs busy when there are few pairs (a 64-particle scene has a few
// hundred).  Row decisions of the hybrid drivers (how many penalty solves
// failed in row iA) are accumulated in LDS in a first pass; the emitting
// pass then evaluates each pair with the method its row requires.  Contacts
// are compacted per chunk with wave ballots and one global atomic per chunk,
// tagged with (tile, rank in tile), and scattered into pair order
// afterwards, so the output order equals the reference's serial emission
// order and does not depend on scheduling or on the tiling.
#include <cstring>
#include <vector>

#include "exact_math.hpp"
#include "gjk.hpp"
#include "pair_range.hpp"
#include "queue_shape.hpp"
#include "runtime.hpp"

namespace dh {

// Longest row the reference's drivers support: per-row stack arrays of
// 10000 entries indexed by 3*iB (bf.cpp:98, penalty.cpp:186, hybrid.cpp:402).
constexpr int kMaxRowTriangles = 3333;

// LDS list of DH_BF candidates that pass the box test (per workgroup), and
// the most triangles per particle whose boxes are staged in LDS.
constexpr int kSurvivors = 1024;
constexpr int kBoxTriangles = kRowBlock;
constexpr int kChunkFlags = 1024;  // chunks of 64 rows an item tests up front

enum DetectError : int { DE_NONE = 0, DE_REF_UB = 1, DE_TOO_LONG = 2 };

// Per-tile counters (tile_stats) and the stats slot each one is summed into;
// DH_BF keeps the first kBfStats only.
enum TileStat : int {
  TS_CHECKS = 0, TS_EVALUATED, TS_CULLED, kBfStats,
  TS_FALLBACK_ROWS = kBfStats, TS_PENALTY_FAILS, TS_BATCH_FAILS, TS_BATCH_SIZE, kTileStats
};

enum StatSlot : int {
  ST_HIST = 0,            // 17 slots
  ST_PENALTY_FAILS = 17,
  ST_BATCH_FAILS = 18,
  ST_BATCH_SIZE = 19,
  ST_CHECKS = 20,
  ST_EVALUATED = 21,
  ST_FALLBACK_ROWS = 22,
  ST_CULLED = 23,  // DH_BF triangle pairs skipped by the box test
  ST_COUNT = 24
};

struct DetectArgs {
  const double* x;
  const double* y;
  const double* z;
  const int* tri_offset;
  const double* eps;
  const int* friction;
  const int* id;
  const int* pairs;
  int npairs;
  dh_contact* temp;  // unordered contacts: pair = tile, pad_ = rank within the tile
  long long cap;
  unsigned long long* counter;  // [0] contacts reserved
  int tiles;                    // row ranges (workgroups) per particle pair
  int* tile_count;              // contacts per (pair, tile), pair-major
  // kTileStats counters per tile (TS_*), summed by k_tile_stats afterwards:
  // one global atomic per workgroup and counter would serialise the launch
  unsigned long long* tile_stats;
  unsigned long long* stats;  // ST_COUNT counters
  int* error;                 // DetectError of the first failing pair
  // When set, the number of pairs is read here (at most npairs, which is then
  // the launch capacity); pairs beyond it record no contacts.
  const long long* npairs_dev;
  // When set, a box per particle (lo xyz, hi xyz) containing its vertices:
  // the broad phase's inflated boxes.  Rows apart from B's particle box are
  // apart from every box of B's triangles, so a block of rows that is all
  // apart is skipped before B's triangles are loaded.
  const double* pbox;
  // With pbox, DH_BF: the particles' bounding spheres (x, y, z, r) of the
  // same broad phase.  A pair whose spheres are apart by more than the
  // margin (and a rounding band) has every triangle pair beyond the margin
  // and is skipped whole (culled), as the reference's engine loop may skip
  // it by its own bounding-sphere test (Engine.cpp:272-295).
  const double* psph;
  // With pbox: the broad phase's boxes of the 64-triangle chunks of the
  // particles with more than kRowBlock triangles (chunk c of particle i at
  // bbox[6 * (tri_offset[i] / 64 + i + c)]).  Rows of a chunk apart from
  // B's particle box are not loaded; a block without a near chunk is
  // skipped.
  const double* bbox;
  int nstats;  // counters per tile: kBfStats (DH_BF) or kTileStats
  // Survivor queue of a DH_BF launch (null: every item solves its own
  // survivors), in segments: one of rcap entries for every wave of
  // k_detect_wave, so that no wave waits for a counter that all share, and
  // behind those the blocks of the pool.  An item that does not fit what is
  // left of its wave's segment takes as many blocks in a row as it needs, which
  // are the wave's segment from then on.  rcount[r] is segment r's number of
  // entries (one of several blocks goes by the first block's number; the
  // others' stays 0).  An item that cannot queue goes to `deferred`, for a
  // launch that runs those items in full, taking its items from item_list.
  int4* queue;  // {item, triangle of A, triangle of B, iA | iB << 16}
  QueueShape shape;
  int most;        // entries of an item that may queue
  unsigned* pool;  // blocks taken of each part, kPoolStride apart
  int* rcount;
  // contacts of the queue's entries, in the entries' order, from the place of
  // the segment's first entry; segment r's number in rcount[segments + r]
  struct QueueRecord* rec;
  int heavy;    // segments with more entries are solved in four parts
  int* rparts;  // a heavy segment's: each part's contacts and rank base
  int* deferred;
  unsigned* ndeferred;
  // Items k_lane_cull leaves for k_detect_wave
  struct WaveItem* wlist;
  unsigned* nwlist;
  const int* item_list;
  const unsigned* nitems_dev;  // with item_list: its length (else the launch's)
  unsigned* item_next;         // counts the items taken after each workgroup's first
  int fp32_screen;             // k_queue_solve screens in binary32 first
  // item_skip[item] != 0: k_chunk_cull culled the item and wrote its
  // counters (a launch of DH_BF without the survivor queue skips it)
  const unsigned char* item_skip;
};

// Triangles of A's rows and B's columns, together, whose boxes a wave of
// k_detect_wave holds in LDS after the tests against the other particle.
constexpr int kWaveBoxes = 160;
constexpr int kWavesPerGroup = 2;    // of k_detect_wave

struct WaveItem {
  int item, pa, pb;
  int oA, oB;      // first triangles of A and of B
  int r0, nrows;   // rows [r0, r0 + nrows) of A
  int nB, chunked; // chunked: A's 64-row chunks have boxes in bbox
  double epsA, epsB;
};

struct QueueRecord {
  int item, tris;  // iA | iB << 16
  int rank;        // among the item's contacts
  int pad_;
  double pq[6];
};

__device__ __forceinline__ Tri<double> load_tri(const DetectArgs& g, int t) {
  Tri<double> r;
  const int b = 3 * t;
#pragma unroll
  for (int k = 0; k < 3; ++k) r.v[k] = {g.x[b + k], g.y[b + k], g.z[b + k]};
  return r;
}

// Mid-phase of DH_BF: true when the triangles' bounding boxes, grown by the
// contact margin, are apart along some axis by more than a rounding band.
// The distance then exceeds the margin, so bf (bf.cpp:125-127) emits no
// contact and the pair need not be solved.  Coordinates that are NaN drop
// out of the boxes; bfSolver's result never comes from them either (its
// strict minimum skips NaN features), so the test stays exact.
__device__ __forceinline__ void tri_box(const Tri<double>& T, double* lo, double* hi) {
  lo[0] = fmin(fmin(T.v[0].x, T.v[1].x), T.v[2].x);
  lo[1] = fmin(fmin(T.v[0].y, T.v[1].y), T.v[2].y);
  lo[2] = fmin(fmin(T.v[0].z, T.v[1].z), T.v[2].z);
  hi[0] = fmax(fmax(T.v[0].x, T.v[1].x), T.v[2].x);
  hi[1] = fmax(fmax(T.v[0].y, T.v[1].y), T.v[2].y);
  hi[2] = fmax(fmax(T.v[0].z, T.v[1].z), T.v[2].z);
}

__device__ __forceinline__ bool boxes_apart(const double* loA, const double* hiA,
                                            const double* loB, const double* hiB, double margin) {
  double gap = -INFINITY, mag = 0.0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    gap = fmax(gap, fmax(loB[q] - hiA[q], loA[q] - hiB[q]));
    mag = fmax(mag, fmax(fmax(fabs(loA[q]), fabs(hiA[q])), fmax(fabs(loB[q]), fabs(hiB[q]))));
  }
  return gap > margin * (1.0 + 0x1p-20) + mag * 0x1p-40;
}

__device__ __forceinline__ bool boxes_apart(const Tri<double>& A, const Tri<double>& B,
                                            double margin) {
  double a[6], b[6];
  tri_box(A, a, a + 3);
  tri_box(B, b, b + 3);
  return boxes_apart(a, a + 3, b, b + 3, margin);
}

struct Pair {
  int pa, pb, oA, oB, nA, nB;
  double epsA, epsB, margin, max_err;
  int fric, idA, idB;
};

__device__ __forceinline__ Pair load_pair(const DetectArgs& g, int k) {
  Pair p;
  p.pa = g.pairs[2 * k];
  p.pb = g.pairs[2 * k + 1];
  p.oA = g.tri_offset[p.pa];
  p.oB = g.tri_offset[p.pb];
  p.nA = g.tri_offset[p.pa + 1] - p.oA;
  p.nB = g.tri_offset[p.pb + 1] - p.oB;
  p.epsA = g.eps[p.pa];
  p.epsB = g.eps[p.pb];
  p.margin = p.epsA + p.epsB;
  p.max_err = (p.epsA + p.epsB) / 16.0;
  p.fric = (g.friction[p.pa] && g.friction[p.pb]) ? 1 : 0;
  p.idA = g.id[p.pa];
  p.idB = g.id[p.pb];
  return p;
}

// The particles' bounding spheres (the broad phase's centre and largest
// vertex distance) apart by more than the margin, with an allowance for the
// rounding of the spheres and of bfSolver's distance: no triangle pair of
// the two particles emits a contact.
__device__ __forceinline__ bool spheres_apart(const DetectArgs& g, const Pair& p) {
  if (!g.psph) return false;
  const double* sa = g.psph + 4 * static_cast<long long>(p.pa);
  const double* sb = g.psph + 4 * static_cast<long long>(p.pb);
  const double dx = sa[0] - sb[0], dy = sa[1] - sb[1], dz = sa[2] - sb[2];
  const double mag = fmax(fmax(fmax(fabs(sa[0]), fabs(sa[1])), fmax(fabs(sa[2]), fabs(sb[0]))),
                          fmax(fabs(sb[1]), fabs(sb[2]))) + sa[3] + sb[3];
  const double reach = sa[3] + sb[3] + p.margin * (1.0 + 0x1p-20) + mag * 0x1p-36;
  return dx * dx + dy * dy + dz * dz > reach * reach;
}

// A triangle's box [lo, hi] apart from a particle's bounding sphere s
// (centre, radius) by more than the margin, with spheres_apart's allowance:
// no triangle of that particle is within the margin of the box's triangle.
__device__ __forceinline__ bool box_sphere_apart(const double* lo, const double* hi,
                                                 const double* s, double margin) {
  double d2 = 0.0, mag = 0.0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double e = fmax(fmax(lo[q] - s[q], s[q] - hi[q]), 0.0);
    d2 += e * e;
    mag = fmax(mag, fmax(fmax(fabs(lo[q]), fabs(hi[q])), fabs(s[q])));
  }
  const double reach = s[3] + margin * (1.0 + 0x1p-20) + (mag + s[3]) * 0x1p-36;
  return d2 > reach * reach;
}

__device__ __forceinline__ bool penalty_pair(const Tri<double>& A, const Tri<double>& B,
                                             double max_err, V3<double>& P, V3<double>& Q) {
  const double x0[4] = {0.33, 0.33, 0.33, 0.33};
  return penalty_fixed(A, B, x0, 4, max_err, P, Q);
}

// False for triangles that DH_BF's box or plane test proves to be further
// apart than the margin.
__device__ __forceinline__ bool may_touch(const Tri<double>& A, const Tri<double>& B,
                                          double margin) {
  return !boxes_apart(A, B, margin) && !plane_apart(A, B, margin);
}

// Row fallback rules.
template <int M>
__device__ __forceinline__ bool row_falls_back(int fails, int nB, double max_err) {
  if (M == DH_HYBRID_TRIANGLE) return fails > 0;
  const double local = fails * max_err;
  if (M == DH_HYBRID_BATCH) return local > (max_err * static_cast<double>(3 * nB)) / 32.0;
  return local > (max_err * static_cast<double>(nB)) / 32;  // *Stat variants
}

template <int M>
__device__ __forceinline__ double final_pair(const DetectArgs& g, const Pair& p, int iA, int iB,
                                             const int* row_fail, int r0, V3<double>& P,
                                             V3<double>& Q) {
  const Tri<double> A = load_tri(g, p.oA + iA);
  const Tri<double> B = load_tri(g, p.oB + iB);
  if (M == DH_BF) {
    bf_solver(A, B, P, Q);
  } else if (M == DH_PENALTY) {
    penalty_pair(A, B, p.max_err, P, Q);
  } else if (M == DH_PENALTY_STAT) {
    penalty_adaptive(A, B, p.max_err, P, Q);
  } else {
    if (row_falls_back<M>(row_fail[iA - r0], p.nB, p.max_err))
      bf_solver(A, B, P, Q);
    else
      penalty_pair(A, B, p.max_err, P, Q);
  }
  return pq_dist(P, Q);
}

__device__ __forceinline__ void make_contact(const Pair& p, int k, int iA, int iB,
                                             const V3<double>& P, const V3<double>& Q,
                                             dh_contact* c) {
  // contactpoint.cpp:116-155
  c->x[0] = (P.x + Q.x) / 2.0;
  c->x[1] = (P.y + Q.y) / 2.0;
  c->x[2] = (P.z + Q.z) / 2.0;
  c->P[0] = P.x; c->P[1] = P.y; c->P[2] = P.z;
  c->Q[0] = Q.x; c->Q[1] = Q.y; c->Q[2] = Q.z;
  c->eps_total = p.epsA + p.epsB;
  const double dist = pq_dist(P, Q);
  c->depth = c->eps_total - dist;
  c->normal[0] = (P.x - Q.x) / dist;
  c->normal[1] = (P.y - Q.y) / dist;
  c->normal[2] = (P.z - Q.z) / dist;
  c->master = p.idA;
  c->slave = p.idB;
  c->penetration = 1;
  c->friction = p.fric;
  c->triA = iA;
  c->triB = iB;
  c->pair = k;
}

// One (particle pair, row range) item of the detection: `item` = pair *
// tiles + tile.  Returns when the item is done; the caller synchronises the
// workgroup before its next item.
template <int M>
__device__ __forceinline__ void detect_item(const DetectArgs& g, const int item) {
  extern __shared__ unsigned char smem[];
  __shared__ int wave_cnt[4];
  __shared__ unsigned long long chunk_base;
  __shared__ unsigned long long local_stats[6];

  const int k = item / g.tiles, tile = item - k * g.tiles;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  unsigned long long* ts = g.tile_stats + static_cast<long long>(item) * g.nstats;
  if (M == DH_BF && g.item_skip && g.item_skip[item]) return;  // k_chunk_cull's
  if (g.npairs_dev && k >= *g.npairs_dev) {
    if (tid == 0) g.tile_count[item] = 0;
    if (tid < g.nstats) ts[tid] = 0;
    return;
  }
  const Pair p = load_pair(g, k);
  const bool is_hybrid = (M == DH_HYBRID_BATCH || M == DH_HYBRID_TRIANGLE ||
                          M == DH_HYBRID_BATCH_STAT || M == DH_HYBRID_TRIANGLE_STAT);
  const bool is_rowstat = (M == DH_HYBRID_BATCH_STAT || M == DH_HYBRID_TRIANGLE_STAT);
  const int rows = (M == DH_HYBRID_TRIANGLE) ? p.nB : p.nA;

  if (M == DH_HYBRID_TRIANGLE && p.nB > p.nA) {
    if (tid == 0) atomicCAS(g.error, DE_NONE, static_cast<int>(DE_REF_UB));
    if (tid == 0) g.tile_count[item] = 0;
    if (tid < g.nstats) ts[tid] = 0;
    return;
  }
  if ((is_hybrid || is_rowstat) && (rows > kMaxRowTriangles || p.nB > kMaxRowTriangles)) {
    if (tid == 0) atomicCAS(g.error, DE_NONE, static_cast<int>(DE_TOO_LONG));
    if (tid == 0) g.tile_count[item] = 0;
    if (tid < g.nstats) ts[tid] = 0;
    return;
  }
  // this workgroup's rows [r0, r1)
  const int r0 = static_cast<int>(static_cast<long long>(tile) * rows / g.tiles);
  const int r1 = static_cast<int>(static_cast<long long>(tile + 1) * rows / g.tiles);
  const int nrows = r1 - r0;
  if (tid < 6) local_stats[tid] = 0;

  int* row_fail = reinterpret_cast<int*>(smem);
  int* row_lastnan = row_fail + kMaxRowTriangles;
  unsigned long long* row_min =
      reinterpret_cast<unsigned long long*>(smem + 2 * kMaxRowTriangles * sizeof(int) + 8);
  // the triangle pairs of this tile: its rows, or, where no pair needs another,
  // chunks of 256, which leave no wave of the last round idle (rows of 80 did
  // for the penalty's 12 tiles of 6,400 pairs: 137 us, 133 us so)
  constexpr bool kFlat = M == DH_PENALTY || M == DH_PENALTY_STAT;
  const PairRange range = kFlat ? pair_range(rows, p.nB, g.tiles, tile)
                                : PairRange{static_cast<long long>(nrows) * p.nB, r0, 0};
  // the pairs of a hybrid tile whose penalty points are within the margin, so
  // that a row which does not fall back is not solved again for the others
  // (a tile of more pairs solves all of them twice)
  constexpr bool kNoted = M == DH_HYBRID_BATCH || M == DH_HYBRID_TRIANGLE;
  constexpr int kNotedPairs = 16384;
  __shared__ unsigned long long close_bits[kNoted ? kNotedPairs / 64 : 1];
  const bool noted = kNoted && range.count <= kNotedPairs;
  // the hybrids' pairs, of at most kMaxRowTriangles rows and columns
  const int f0 = is_hybrid ? r0 * p.nB : 0, total = is_hybrid ? nrows * p.nB : 0;

  if (is_hybrid) {
    for (int r = tid; r < nrows; r += 256) {
      row_fail[r] = 0;
      if (is_rowstat) {
        row_lastnan[r] = -1;
        row_min[r] = ~0ull;
      }
    }
    __syncthreads();
    // pass 1: penalty on every pair, failures per row
    for (int f = f0 + tid; f < f0 + total; f += 256) {
      const int iA = f / p.nB, iB = f - iA * p.nB;
      const Tri<double> A = load_tri(g, p.oA + iA);
      const Tri<double> B = load_tri(g, p.oB + iB);
      V3<double> P, Q;
      if (penalty_pair(A, B, p.max_err, P, Q)) atomicAdd(&row_fail[iA - r0], 1);
      if (noted) {
        const unsigned long long m = __ballot(pq_dist(P, Q) < p.margin);
        if (lane == 0) close_bits[(f - f0) >> 6] = m;
      }
    }
    __syncthreads();
    if (tid == 0) {
      unsigned long long fb = 0, fails = 0, bfails = 0;
      for (int r = 0; r < nrows; ++r) {
        fails += row_fail[r];
        if (row_falls_back<M>(row_fail[r], p.nB, p.max_err)) {
          fb++;
          bfails++;
        }
      }
      local_stats[0] = fb;
      local_stats[1] = fails;
      local_stats[2] = bfails;
    }
  }
  if (is_rowstat) {
    // pass 2: last NaN distance per row; pass 3: minimum after it
    // (std::min(d, minD) semantics of hybrid.cpp:316-318)
    for (int f = f0 + tid; f < f0 + total; f += 256) {
      const int iA = f / p.nB, iB = f - iA * p.nB;
      V3<double> P, Q;
      const double d = final_pair<M>(g, p, iA, iB, row_fail, r0, P, Q);
      if (d != d) atomicMax(&row_lastnan[iA - r0], iB);
    }
    __syncthreads();
    for (int f = f0 + tid; f < f0 + total; f += 256) {
      const int iA = f / p.nB, iB = f - iA * p.nB;
      if (iB <= row_lastnan[iA - r0]) continue;
      V3<double> P, Q;
      const double d = final_pair<M>(g, p, iA, iB, row_fail, r0, P, Q);
      atomicMin(&row_min[iA - r0], static_cast<unsigned long long>(__double_as_longlong(d)));
    }
    __syncthreads();
  }

  // Emission of one chunk of 256 candidates (in row-major order across
  // chunks): block prefix over the emitting lanes, one global atomic for the
  // chunk's slots, rank within the tile in pad_.
  unsigned long long running = 0;
  bool far_pair = false;
  unsigned culled = 0;  // of a lane; a whole pair's are counted at the end
  auto emit_chunk = [&](bool emit, int iA, int iB, const V3<double>& P, const V3<double>& Q) {
    const unsigned long long mask = __ballot(emit);
    const int pre = lane_prefix(mask);
    if (lane == 0) wave_cnt[wave] = __popcll(mask);
    __syncthreads();
    int off = 0, cnt = 0;
    for (int w = 0; w < 4; ++w) {
      off += (w < wave) ? wave_cnt[w] : 0;
      cnt += wave_cnt[w];
    }
    if (tid == 0 && cnt > 0) chunk_base = atomicAdd(g.counter, static_cast<unsigned long long>(cnt));
    __syncthreads();
    if (emit) {
      const unsigned long long slot = chunk_base + off + pre;
      if (slot < static_cast<unsigned long long>(g.cap)) {
        dh_contact c;
        make_contact(p, k, iA, iB, P, Q, &c);
        c.pair = item;  // the tile, until the scatter
        c.pad_ = static_cast<int>(running + off + pre);
        g.temp[slot] = c;
      }
    }
    running += cnt;
    __syncthreads();
  };

  if (M == DH_BF) {
    // Box test first, survivors compacted in row-major order into LDS, then
    // solved 256 at a time, so that no lane idles beside a culled pair.  When
    // B's triangle boxes fit in LDS they are staged there once, the tile's
    // rows are staged in blocks of up to kBoxTriangles (a large A such as a
    // funnel or a wall takes several blocks, in row order), and only rows
    // whose box meets the union of B's boxes and columns whose box meets the
    // union of the block's rows are paired (the union test implies the pair
    // test, so nothing else changes).  A larger B takes one unstaged pass.
    __shared__ int surv[kSurvivors];
    __shared__ double boxes[2 * kBoxTriangles * 6];
    __shared__ int act[2 * kBoxTriangles];  // active rows (block-relative), then columns
    __shared__ double uni[2][6];            // union of the block's row boxes, of B's boxes
    __shared__ double red[4][12];
    __shared__ int nact[2];
    __shared__ unsigned char row_far[kBoxTriangles];  // row in a chunk apart from B
    __shared__ unsigned char chunk_near[kChunkFlags];  // the item's chunks against B's box
    const bool staged = p.nB <= kBoxTriangles;  // block-uniform
    // an unstaged block's pairs are numbered in 32 bits
    const int most = p.nB > 0 ? (1 << 30) / p.nB : 1 << 30;
    const int blk = staged ? kBoxTriangles : (nrows < most ? (nrows > 0 ? nrows : 1) : (most > 0 ? most : 1));
    bool b_staged = false;  // B's boxes are loaded on the first block that needs them
    // the whole pair beyond the margin by its bounding spheres
    far_pair = spheres_apart(g, p);
    // A in chunks of 64 rows with their boxes (a wall or a funnel): every
    // chunk of the item tested against B's particle box once, up front
    const bool chunked = staged && g.bbox && g.pbox && p.nA > kRowBlock;
    const double* pbB = g.pbox ? g.pbox + 6 * static_cast<long long>(p.pb) : nullptr;
    // row r of A (particle-relative) lies in a chunk apart from B's box
    auto chunk_far = [&](int r) {
      const double* cb = g.bbox + 6 * (static_cast<long long>(p.oA / 64) + p.pa + r / 64);
      return boxes_apart(cb, cb + 3, pbB, pbB + 3, p.margin);
    };
    const int c_first = r0 / 64;
    const bool flagged = chunked && nrows > 0 && (r0 + nrows - 1) / 64 - c_first < kChunkFlags;
    if (flagged && !far_pair) {
      for (int c = tid; c <= (r0 + nrows - 1) / 64 - c_first; c += 256)
        chunk_near[c] = chunk_far(64 * (c_first + c)) ? 0 : 1;
      __syncthreads();
    }
    auto row_chunk_far = [&](int r) {
      return flagged ? chunk_near[r / 64 - c_first] == 0 : chunk_far(r);
    };
    for (int rb = 0; !far_pair && rb < nrows; rb += blk) {
      const int rs = r0 + rb;  // first row of the block
      const int nrb = nrows - rb < blk ? nrows - rb : blk;
      int nra = nrb, nca = p.nB;
      if (flagged) {
        // the same flags in every thread: no barrier
        bool any_near = false;
        for (int c = rs / 64; c <= (rs + nrb - 1) / 64; ++c)
          any_near = any_near || chunk_near[c - c_first] != 0;
        if (!any_near) {  // every chunk of the block is apart
          culled += tid == 0 ? nrb * p.nB : 0;
          continue;
        }
      } else if (chunked) {
        bool any_near = false;
        for (int c = rs / 64 + tid; c <= (rs + nrb - 1) / 64; c += 256)
          any_near = any_near || !chunk_far(64 * c);
        if (!__syncthreads_or(any_near)) {  // every chunk of the block is apart
          culled += tid == 0 ? nrb * p.nB : 0;
          continue;
        }
      }
      if (staged) {
        bool near = false;
        for (int t = tid; t < nrb; t += 256) {
          const bool far = chunked && row_chunk_far(rs + t);
          row_far[t] = far ? 1 : 0;
          if (far) continue;  // its box is never read
          double* b = boxes + 6 * t;
          tri_box(load_tri(g, p.oA + rs + t), b, b + 3);
          if (g.pbox) near = near || !boxes_apart(b, b + 3, pbB, pbB + 3, p.margin);
        }
        if (g.pbox && !__syncthreads_or(near)) {
          // every row of the block misses B's particle box
          culled += tid == 0 ? nrb * p.nB : 0;
          continue;
        }
        if (!b_staged) {
          for (int t = tid; t < p.nB; t += 256) {
            double* b = boxes + 6 * (kBoxTriangles + t);
            tri_box(load_tri(g, p.oB + t), b, b + 3);
          }
          b_staged = true;
        }
        __syncthreads();
        // unions: lanes over strided boxes, then waves, then the block
        double u[12];
        for (int q = 0; q < 3; ++q) {
          u[q] = u[6 + q] = INFINITY;
          u[3 + q] = u[9 + q] = -INFINITY;
        }
        for (int t = tid; t < nrb; t += 256)
          if (!row_far[t])
            for (int q = 0; q < 3; ++q) {
              u[q] = fmin(u[q], boxes[6 * t + q]);
              u[3 + q] = fmax(u[3 + q], boxes[6 * t + 3 + q]);
            }
        for (int t = tid; t < p.nB; t += 256)
          for (int q = 0; q < 3; ++q) {
            u[6 + q] = fmin(u[6 + q], boxes[6 * (kBoxTriangles + t) + q]);
            u[9 + q] = fmax(u[9 + q], boxes[6 * (kBoxTriangles + t) + 3 + q]);
          }
        for (int o = 32; o > 0; o >>= 1)
          for (int q = 0; q < 12; ++q) {
            const double v = __shfl_xor(u[q], o);
            u[q] = ((q % 6) < 3) ? fmin(u[q], v) : fmax(u[q], v);
          }
        if (lane == 0)
          for (int q = 0; q < 12; ++q) red[wave][q] = u[q];
        __syncthreads();
        if (tid < 12) {
          double v = red[0][tid];
          for (int w = 1; w < 4; ++w) v = ((tid % 6) < 3) ? fmin(v, red[w][tid]) : fmax(v, red[w][tid]);
          uni[tid / 6][tid % 6] = v;
        }
        if (tid < 2) nact[tid] = 0;
        __syncthreads();
        // ordered lists of active rows and columns
        for (int side = 0; side < 2; ++side) {
          const int cnt_all = side == 0 ? nrb : p.nB;
          const double* other = uni[1 - side];
          for (int t0 = 0; t0 < cnt_all; t0 += 256) {
            const int t = t0 + tid;
            bool on = false;
            if (t < cnt_all && !(side == 0 && row_far[t])) {
              const double* b = boxes + 6 * (side == 0 ? t : kBoxTriangles + t);
              on = !boxes_apart(b, b + 3, other, other + 3, p.margin);
            }
            const unsigned long long m = __ballot(on);
            if (lane == 0) wave_cnt[wave] = __popcll(m);
            __syncthreads();
            int off = 0, cnt = 0;
            for (int w = 0; w < 4; ++w) {
              off += (w < wave) ? wave_cnt[w] : 0;
              cnt += wave_cnt[w];
            }
            if (on) act[side * kBoxTriangles + nact[side] + off + lane_prefix(m)] = t;
            __syncthreads();
            if (tid == 0) nact[side] += cnt;
            __syncthreads();
          }
        }
        nra = nact[0];
        nca = nact[1];
      }
      // candidate fe in [0, nra * nca): row-major over the active rows and columns
      auto pair_of = [&](int fe, int& iA, int& iB) {
        const int ra = fe / nca, cb = fe - ra * nca;
        iA = staged ? rs + act[ra] : rs + ra;
        iB = staged ? act[kBoxTriangles + cb] : cb;
      };
      const int tested = nra * nca;
      culled += tid == 0 ? nrb * p.nB - tested : 0;
      for (int fpos = 0; fpos < tested;) {
        int nl = 0;
        while (fpos < tested && nl <= kSurvivors - 256) {
          const int fe = fpos + tid;
          bool keep = false;
          if (fe < tested) {
            int iA, iB;
            pair_of(fe, iA, iB);
            if (staged) {
              const double* a = boxes + 6 * (iA - rs);
              const double* b = boxes + 6 * (kBoxTriangles + iB);
              keep = !boxes_apart(a, a + 3, b, b + 3, p.margin);
            } else {
              keep = !boxes_apart(load_tri(g, p.oA + iA), load_tri(g, p.oB + iB), p.margin);
            }
            culled += keep ? 0 : 1;
          }
          const unsigned long long m = __ballot(keep);
          if (lane == 0) wave_cnt[wave] = __popcll(m);
          __syncthreads();
          int off = 0, cnt = 0;
          for (int w = 0; w < 4; ++w) {
            off += (w < wave) ? wave_cnt[w] : 0;
            cnt += wave_cnt[w];
          }
          if (keep) surv[nl + off + lane_prefix(m)] = fe;
          nl += cnt;
          fpos += 256;
          __syncthreads();
        }
        // the survivors that a triangle plane separates by more than the
        // margin (and, with the binary32 screen, those it proves far) drop
        // out; the rest are compacted in place (order kept) for the
        // binary64 solve.  (The edge-pair axes of the queue paths do not
        // pay here: an item keeps one wave's bfSolver round as long as a
        // survivor is left, whatever their number.)
        int n2 = 0;
        for (int b = 0; b < nl; b += 256) {
          const int e = b + tid;
          int v = 0;
          bool keep2 = false;
          if (e < nl) {
            v = surv[e];
            int iA, iB;
            pair_of(v, iA, iB);
            const Tri<double> A = load_tri(g, p.oA + iA), B = load_tri(g, p.oB + iB);
            keep2 = !plane_apart(A, B, p.margin) &&
                    !(g.fp32_screen && screened_far(A, B, p.margin));
          }
          const unsigned long long m = __ballot(keep2);
          if (lane == 0) wave_cnt[wave] = __popcll(m);
          __syncthreads();
          int off = 0, cnt = 0;
          for (int w = 0; w < 4; ++w) {
            off += (w < wave) ? wave_cnt[w] : 0;
            cnt += wave_cnt[w];
          }
          if (keep2) surv[n2 + off + lane_prefix(m)] = v;
          n2 += cnt;
          __syncthreads();
        }
        nl = n2;
        for (int b = 0; b < nl; b += 256) {
          const int e = b + tid;
          bool emit = false;
          V3<double> P = {0, 0, 0}, Q = {0, 0, 0};
          int iA = 0, iB = 0;
          if (e < nl) {
            pair_of(surv[e], iA, iB);
            bf_solver_general(load_tri(g, p.oA + iA), load_tri(g, p.oB + iB), P, Q);
            emit = pq_dist(P, Q) <= p.margin;
          }
          emit_chunk(emit, iA, iB, P, Q);
        }
      }
      // the next block overwrites the row boxes and the active lists
      __syncthreads();
    }
  } else {
    PairWalk at(range, p.nB, tid);
    for (long long left = range.count; left > 0; left -= kPairChunk) {
      const int f = static_cast<int>(range.count - left) + tid;  // read where the tile is noted
      bool emit = false;
      V3<double> P = {0, 0, 0}, Q = {0, 0, 0};
      const int iA = at.iA, iB = at.iB;
      if (tid < left) {
        if (M == DH_PENALTY_STAT) {
          const Tri<double> A = load_tri(g, p.oA + iA);
          const Tri<double> B = load_tri(g, p.oB + iB);
          const int its = penalty_adaptive(A, B, p.max_err, P, Q);
          atomicAdd(&g.stats[ST_HIST + (its < 0 ? 0 : its)], 1ull);
          const double d = pq_dist(P, Q);
          emit = (3 * iB < p.nB) && (d <= p.margin);
        } else if (noted && !(row_falls_back<M>(row_fail[iA - r0], p.nB, p.max_err)
                                  ? may_touch(load_tri(g, p.oA + iA), load_tri(g, p.oB + iB),
                                              p.margin)
                                  : (close_bits[f >> 6] >> (f & 63)) & 1)) {
          // not within the margin
        } else {
          const double d = final_pair<M>(g, p, iA, iB, row_fail, r0, P, Q);
          if (is_rowstat) {
            double mn;
            if (row_lastnan[iA - r0] == p.nB - 1) {
              mn = __longlong_as_double(0x7ff8000000000000ll);
            } else {
              mn = __longlong_as_double(static_cast<long long>(row_min[iA - r0]));
              if (row_lastnan[iA - r0] < 0) mn = (1E99 < mn) ? 1E99 : mn;
            }
            emit = (d <= mn) && (d < p.margin);
          } else {
            emit = d < p.margin;
          }
        }
      }
      emit_chunk(emit, iA, iB, P, Q);
      at.next(p.nB);
    }
  }
  if (M == DH_BF) {
    // slot 3 of local_stats (zeroed at the start, unused by BF otherwise)
    unsigned long long sum = far_pair && tid == 0 ? range.count : culled;
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) atomicAdd(&local_stats[3], sum);
    __syncthreads();
  }
  if (tid == 0) {
    g.tile_count[item] = static_cast<int>(running);
    // evaluations the reference performs: every pair once, plus bfSolver
    // again over each fallback row (sums over the tiles)
    const unsigned long long evals =
        static_cast<unsigned long long>(range.count) +
        (is_hybrid ? local_stats[0] * static_cast<unsigned long long>(p.nB) : 0ull);
    ts[TS_CHECKS] = tile == 0 ? static_cast<unsigned long long>(p.nA) * p.nB : 0ull;
    ts[TS_EVALUATED] = evals;
    ts[TS_CULLED] = M == DH_BF ? local_stats[3] : 0ull;
    if (M != DH_BF) {
      ts[TS_FALLBACK_ROWS] = is_hybrid ? local_stats[0] : 0ull;
      ts[TS_PENALTY_FAILS] = is_rowstat ? local_stats[1] : 0ull;
      ts[TS_BATCH_FAILS] = is_rowstat ? local_stats[2] : 0ull;
      ts[TS_BATCH_SIZE] = is_rowstat ? static_cast<unsigned long long>(nrows) * p.nB : 0ull;
    }
  }
}

// Persistent over the items: workgroup b takes items b, b + gridDim.x, ...
// (with as many workgroups as items, one each), or with item_next the next one
// that no workgroup has yet.  Pairs of very uneven cost
// (a 2,048-triangle funnel against 20-triangle particles) share the
// workgroups of one launch.  The brute force is held to 168 registers
// (three waves per SIMD; a few spill), which its latency-bound item loop
// needs more than the registers.
template <int M>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(M == DH_BF ? 3 : 1))) void k_detect(DetectArgs g, int items) {
  if (g.item_list && g.nitems_dev && static_cast<int>(*g.nitems_dev) < items)
    items = static_cast<int>(*g.nitems_dev);
  __shared__ int next;
  for (int t = blockIdx.x; t < items;) {
    detect_item<M>(g, g.item_list ? g.item_list[t] : t);
    __syncthreads();  // the next item reuses the workgroup's LDS
    if (g.item_next) {
      if (threadIdx.x == 0) next = static_cast<int>(gridDim.x + atomicAdd(g.item_next, 1u));
      __syncthreads();
      t = next;
    } else {
      t += gridDim.x;
    }
  }
}

// One wave per item, before a DH_BF launch without the survivor queue, on
// scenes with particles of more than kRowBlock triangles (walls, funnels):
// an item whose A is cut in chunks of 64 rows is culled when no row of a
// chunk near B's particle box is itself near it, with the counters
// detect_item would write (its blocks would all be skipped).  The test is
// detect_item's chunk and row tests, without its workgroup barriers.
// item_skip[item] = 1 marks the culled and dead items.
__global__ __launch_bounds__(256) void k_chunk_cull(DetectArgs g, int items,
                                                    unsigned char* __restrict__ skip) {
  const int lane = threadIdx.x & 63;
  const int nw = static_cast<int>(gridDim.x) * 4;
  for (int item = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6);
       item < items; item += nw) {
    const int k = item / g.tiles, tile = item - k * g.tiles;
    unsigned long long* ts = g.tile_stats + static_cast<long long>(item) * g.nstats;
    if (g.npairs_dev && k >= *g.npairs_dev) {
      if (lane == 0) {
        g.tile_count[item] = 0;
        skip[item] = 1;
      }
      if (lane < g.nstats) ts[lane] = 0;
      continue;
    }
    const Pair p = load_pair(g, k);
    const int r0 = static_cast<int>(static_cast<long long>(tile) * p.nA / g.tiles);
    const int r1 = static_cast<int>(static_cast<long long>(tile + 1) * p.nA / g.tiles);
    const bool chunked = p.nB <= kBoxTriangles && g.bbox && g.pbox && p.nA > kRowBlock;
    bool near = !(chunked && r1 > r0);
    if (!near) {
      const double* pbB = g.pbox + 6 * static_cast<long long>(p.pb);
      const int c_last = (r1 - 1) / 64;
      for (int c0 = r0 / 64; c0 <= c_last && !near; c0 += 64) {
        const int c = c0 + lane;
        bool cn = false;
        if (c <= c_last) {
          const double* cb = g.bbox + 6 * (static_cast<long long>(p.oA / 64) + p.pa + c);
          cn = !boxes_apart(cb, cb + 3, pbB, pbB + 3, p.margin);
        }
        unsigned long long m = __ballot(cn);
        while (m && !near) {
          const int cc = c0 + __builtin_ctzll(m);
          m &= m - 1;
          const int r = 64 * cc + lane;
          bool rn = false;
          if (r >= r0 && r < r1) {
            double lo[3], hi[3];
            tri_box(load_tri(g, p.oA + r), lo, hi);
            rn = !boxes_apart(lo, hi, pbB, pbB + 3, p.margin);
          }
          near = __ballot(rn) != 0;
        }
      }
    }
    if (lane == 0) {
      skip[item] = near ? 0 : 1;
      if (!near) {
        const unsigned long long total = static_cast<unsigned long long>(r1 - r0) * p.nB;
        g.tile_count[item] = 0;
        ts[TS_CHECKS] = tile == 0 ? static_cast<unsigned long long>(p.nA) * p.nB : 0ull;
        ts[TS_EVALUATED] = total;
        ts[TS_CULLED] = total;
      }
    }
  }
}

// Rows a lane tests alone in k_lane_cull.
constexpr int kLaneRows = 16;

// Up to this many items, in workgroups of 256: more CUs share the lanes'
// scattered loads (4,600 items 13.5 -> 8.3 us); above, the atomic per
// workgroup counts for more.
constexpr int kFewItems = 65536;

// One lane per item, before k_detect_wave: an item whose particles' bounding
// spheres are apart by more than the margin (diagonal neighbours in a
// packing), or with at most kLaneRows rows whose rows' boxes all miss B's
// particle box (grown by the margin: a wall of few triangles against the many
// particles inside it), is culled here, with the counters the mid-phase would
// write.  The others are listed for k_detect_wave with what it needs of them
// (its loads of triangles then wait for one load, not for three in a row).
// Items whose triangle numbers do not fit a queue entry are deferred.  One
// atomic per workgroup and list: one per wave took most of the 43 us that the
// hopper's 3.8e5 items spent here (11 us now).
__global__ __launch_bounds__(1024) void k_lane_cull(DetectArgs g, int items) {
  __shared__ unsigned wave_cnt[16], base;
  const int tid = static_cast<int>(threadIdx.x);
  const int item = blockIdx.x * blockDim.x + tid;
  const int wave = tid >> 6;
  bool listed = false;
  WaveItem it = {};
  if (item < items) {
    const int k = item / g.tiles, tile = item - k * g.tiles;
    unsigned long long* ts = g.tile_stats + static_cast<long long>(item) * g.nstats;
    g.tile_count[item] = 0;
    if (!(g.npairs_dev && k >= *g.npairs_dev)) {
      const Pair p = load_pair(g, k);
      const int r0 = static_cast<int>(static_cast<long long>(tile) * p.nA / g.tiles);
      const int r1 = static_cast<int>(static_cast<long long>(tile + 1) * p.nA / g.tiles);
      const int nrows = r1 - r0;
      const unsigned long long total = static_cast<unsigned long long>(nrows) * p.nB;
      bool near = !(g.pbox && nrows <= kLaneRows);
      if (spheres_apart(g, p)) {
        near = false;  // culled whole
      } else if (!near) {
        const double* pb = g.pbox + 6 * static_cast<long long>(p.pb);
        for (int t = 0; t < nrows && !near; ++t) {
          double lo[3], hi[3];
          tri_box(load_tri(g, p.oA + r0 + t), lo, hi);
          near = !boxes_apart(lo, hi, pb, pb + 3, p.margin);
        }
      }
      ts[TS_CHECKS] = tile == 0 ? static_cast<unsigned long long>(p.nA) * p.nB : 0ull;
      ts[TS_EVALUATED] = total;
      ts[TS_CULLED] = total;  // a listed item's own kernel writes its count
      if (near && total > 0) {
        listed = p.nA < 65536 && p.nB < 65536;
        if (!listed) g.deferred[atomicAdd(g.ndeferred, 1u)] = item;
      }
      it = {item, p.pa, p.pb, p.oA, p.oB, r0, nrows, p.nB,
            g.pbox && g.bbox && p.nA > kRowBlock ? 1 : 0, p.epsA, p.epsB};
    }
  }
  const unsigned long long m = __ballot(listed);
  if ((tid & 63) == 0) wave_cnt[wave] = static_cast<unsigned>(__popcll(m));
  __syncthreads();
  if (tid == 0) {
    unsigned n = 0;
    for (unsigned w = 0; w < blockDim.x / 64; ++w) {
      const unsigned c = wave_cnt[w];
      wave_cnt[w] = n;
      n += c;
    }
    base = n ? atomicAdd(g.nwlist, n) : 0u;
  }
  __syncthreads();
  if (listed) g.wlist[base + wave_cnt[wave] + lane_prefix(m)] = it;
}

// The largest gap between two boxes along an axis.
__device__ __forceinline__ double box_gap(const double* loA, const double* hiA, const double* loB,
                                          const double* hiB) {
  double gap = -INFINITY;
#pragma unroll
  for (int q = 0; q < 3; ++q) gap = fmax(gap, fmax(loB[q] - hiA[q], loA[q] - hiB[q]));
  return gap;
}

// The mid-phase of DH_BF, one wave per listed item and no workgroup barrier:
// the boxes of A's rows and B's columns that lie within the margin of the
// other particle's box and bounding sphere are kept, in order, in the wave's
// LDS (the rows of a large A chunk by chunk, those of far chunks unread); the
// pairs of kept rows and columns whose boxes are within the margin are
// appended, in row-major order, to the wave's segment of the survivor queue.
// Items with more than kWaveBoxes kept rows and columns, or more survivors
// than an item may queue or the pool has left, are deferred to the full
// kernel.  The survivors are fewer than detect_item's box test leaves (that one
// does not know the bounding spheres), so pairs_culled depends on the path an
// item took; the contacts do not.
// It is bound by the latency of an item's loads, so it holds little: 16 waves
// per CU.  Separating axes are tested in k_queue_solve instead, with every
// lane busy (here they took 161 registers, 9 waves per CU, for some 10 to 40
// survivors at a time), and the other particle's box from the broad phase
// takes the place of the union of its triangles' boxes (144 lane shuffles per
// item).  What it cost before was an atomic per item on one queue counter,
// some 10 ns each: 610 us for the hopper's 1.9e5 pairs, 87 us with a segment
// per wave (8 workgroups per CU; 6 per CU: 100 us).
__global__ __launch_bounds__(64 * kWavesPerGroup, 4) void k_detect_wave(DetectArgs g) {
  __shared__ double boxes[kWavesPerGroup][kWaveBoxes * 6];
  __shared__ unsigned short act[kWavesPerGroup][kWaveBoxes];
  // of at most kWaveBoxes / 2 rows by as many columns
  __shared__ unsigned long long rounds[kWavesPerGroup][kWaveBoxes * kWaveBoxes / 256 + 1];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  double* bx = boxes[w];
  const int region = blockIdx.x * kWavesPerGroup + w;
  int segment = region, cap = g.shape.rcap, used = 0;
  int4* queue = g.queue + static_cast<long long>(region) * g.shape.rcap;
  bool dry = false;  // the pool has nothing left
  const int nw = static_cast<int>(*g.nwlist);
  for (int j = region; j < nw; j += gridDim.x * kWavesPerGroup) {
    const WaveItem it = g.wlist[j];
    const double margin = it.epsA + it.epsB;
    // what the rows (side 0) and the columns (side 1) are tested against: the
    // other particle's box, and how much of the margin lies in it already
    double other[2][6], in[2] = {0.0, 0.0};
    if (g.pbox) {
      in[0] = it.epsB;
      in[1] = it.epsA;
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        other[0][q] = g.pbox[6 * static_cast<long long>(it.pb) + q];
        other[1][q] = g.pbox[6 * static_cast<long long>(it.pa) + q];
      }
    } else {  // the unions of the triangles' boxes
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        const int n = side == 0 ? it.nB : it.nrows;
        const int t0 = side == 0 ? it.oB : it.oA + it.r0;
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int t = lane; t < n; t += 64) {
          double l[3], h[3];
          tri_box(load_tri(g, t0 + t), l, h);
          for (int q = 0; q < 3; ++q) {
            lo[q] = fmin(lo[q], l[q]);
            hi[q] = fmax(hi[q], h[q]);
          }
        }
        for (int o = 32; o > 0; o >>= 1)
          for (int q = 0; q < 3; ++q) {
            lo[q] = fmin(lo[q], __shfl_xor(lo[q], o));
            hi[q] = fmax(hi[q], __shfl_xor(hi[q], o));
          }
        for (int q = 0; q < 3; ++q) {
          other[side][q] = lo[q];
          other[side][3 + q] = hi[q];
        }
      }
    }
    // boxes apart by more than `reach` along an axis: boxes_apart's test with
    // the largest coordinate of either particle in its rounding band
    double mag = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) mag = fmax(mag, fmax(fabs(other[0][q]), fabs(other[1][q])));
    const double reach = margin * (1.0 + 0x1p-20) + mag * 0x1p-40;
    if (margin > 0.0 && mag * 0x1p-26 > margin) {
      // coordinates of more than 13 km at a margin of 0.2 mm: particles that have
      // grown past all bounds, as an unstable run's do, keep a fifth of their
      // pairs and more through all tests, and k_detect takes those with full
      // lanes (lattice after 1,000 such steps: 143 us, 310 through the queue)
      if (lane == 0) g.deferred[atomicAdd(g.ndeferred, 1u)] = it.item;
      continue;
    }
    // keeps the triangles of [t, t + 64) and below `end` that are on side's
    // own; false when the LDS is full
    int kept = 0;
    auto scan = [&](int side, int t0, int t, int end) {
      const double* sph =
          g.psph ? g.psph + 4 * static_cast<long long>(side == 0 ? it.pb : it.pa) : nullptr;
      const double far = reach + mag * 0x1p-40 - in[side];
      const int i = t + lane;
      double lo[3], hi[3];
      tri_box(load_tri(g, t0 + (i < end ? i : end - 1)), lo, hi);
      const bool on = i < end && !(box_gap(lo, hi, other[side], other[side] + 3) > far) &&
                      !(sph && box_sphere_apart(lo, hi, sph, margin));
      const unsigned long long m = __ballot(on);
      const int at = kept + lane_prefix(m);
      kept += __popcll(m);
      if (kept > kWaveBoxes) return false;
      if (on) {
        double* d = bx + 6 * at;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          d[q] = lo[q];
          d[3 + q] = hi[q];
        }
        act[w][at] = static_cast<unsigned short>(i);
      }
      return true;
    };
    bool fits = true;
    const int r1 = it.r0 + it.nrows;
    if (it.chunked) {
      for (int c0 = it.r0 / 64; c0 <= (r1 - 1) / 64 && fits; c0 += 64) {
        const int c = c0 + lane;
        bool cn = false;
        if (c <= (r1 - 1) / 64) {
          const double* cb = g.bbox + 6 * (static_cast<long long>(it.oA / 64) + it.pa + c);
          cn = !boxes_apart(cb, cb + 3, other[0], other[0] + 3, margin);
        }
        for (unsigned long long m = __ballot(cn); m && fits; m &= m - 1) {
          const int r = 64 * (c0 + __builtin_ctzll(m));
          // rows of the chunk before r0 belong to the tile before
          const int lo = r < it.r0 ? it.r0 : r, hi = r + 64 < r1 ? r + 64 : r1;
          fits = scan(0, it.oA, lo, hi);
        }
      }
    } else {
      for (int r = it.r0; r < r1 && fits; r += 64) fits = scan(0, it.oA, r, r1);
    }
    const int na = kept;
    if (na > 0 && fits && (it.chunked || na + it.nB > kWaveBoxes)) {
      // the columns might not fit: they are tested against the union of the
      // kept rows' boxes instead of A's (a funnel's box holds every particle)
      wave_lds_fence();
      double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
      for (int t = lane; t < na; t += 64)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          lo[q] = fmin(lo[q], bx[6 * t + q]);
          hi[q] = fmax(hi[q], bx[6 * t + 3 + q]);
        }
      for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          lo[q] = fmin(lo[q], __shfl_xor(lo[q], o));
          hi[q] = fmax(hi[q], __shfl_xor(hi[q], o));
        }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        other[1][q] = lo[q];
        other[1][3 + q] = hi[q];
      }
      in[1] = 0.0;
    }
    for (int t = 0; t < it.nB && fits && na > 0; t += 64) fits = scan(1, it.oB, t, it.nB);
    const int nc = kept - na, tested = na * nc;
    wave_lds_fence();
    // Survivors in row-major order over the kept rows and columns, 64 pairs a
    // round: put() writes a round's.  The rounds' survivors are kept for an item
    // that turns out not to fit and is written again, to blocks of the pool that
    // hold it.
    const int step_r = nc > 0 ? 64 / nc : 0, step_c = 64 - step_r * nc;
    int ra = nc > 0 ? lane / nc : 0, cb = lane - ra * nc;
    auto put = [&](unsigned long long m, int at) {
      at += lane_prefix(m);
      if ((m >> lane & 1) && at < cap) {
        const int r = act[w][ra], c = act[w][na + cb];
        queue[at] = make_int4(it.item, it.oA + r, it.oB + c,
                              static_cast<int>(static_cast<unsigned>(r) |
                                               (static_cast<unsigned>(c) << 16)));
      }
      ra += step_r;
      cb += step_c;
      if (cb >= nc) {
        cb -= nc;
        ++ra;
      }
    };
    int S = 0;
    if (fits)
      for (int f = lane, k = 0; f - lane < tested; f += 64, ++k) {
        bool keep = false;
        if (f < tested) {
          const double* a = bx + 6 * ra;
          const double* b = bx + 6 * (na + cb);
          keep = !(box_gap(a, a + 3, b, b + 3) > reach);
        }
        const unsigned long long m = __ballot(keep);
        if (lane == 0) rounds[w][k] = m;
        put(m, used + S);
        S += __popcll(m);
      }
    if (used + S > cap && S <= g.most && !dry) {
      const int n = (S + g.shape.block - 1) / g.shape.block;
      int first = -1, part = 0;
      while (first < 0) {
        // the parts with room, from the workgroup's own on
        const int q = (static_cast<int>(blockIdx.x) + lane) % kPoolParts;
        const bool room = lane < kPoolParts &&
                          static_cast<int>(__hip_atomic_load(&g.pool[kPoolStride * q], __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT)) + n <= g.shape.blocks;
        const unsigned long long m = __ballot(room);
        if (!m) break;
        part = __shfl(q, __builtin_ctzll(m));
        if (lane == 0) first = static_cast<int>(atomicAdd(&g.pool[kPoolStride * part], static_cast<unsigned>(n)));
        first = __shfl(first, 0);
        // another wave took them: the count only grows, so the loop ends
        if (first + n > g.shape.blocks) first = -1;
      }
      dry = first < 0;
      if (!dry) {
        if (lane == 0) g.rcount[segment] = used;
        segment = g.shape.pool_segment(part, first);
        queue = g.queue + g.shape.place(segment);
        cap = n * g.shape.block;
        used = 0;
        ra = lane / nc;
        cb = lane - ra * nc;
        wave_lds_fence();
        for (int k = 0, at = 0; 64 * k < tested; ++k) {
          const unsigned long long m = rounds[w][k];
          put(m, at);
          at += __popcll(m);
        }
      }
    }
    if (!fits || used + S > cap) {
      if (lane == 0) g.deferred[atomicAdd(g.ndeferred, 1u)] = it.item;
    } else {
      used += S;
      if (lane == 0)
        g.tile_stats[static_cast<long long>(it.item) * g.nstats + TS_CULLED] =
            static_cast<unsigned long long>(it.nrows) * it.nB - S;
    }
    wave_lds_fence();  // the next item overwrites the wave's LDS
  }
  if (lane == 0) g.rcount[segment] = used;
}

// The stats slot of a tile counter.
__device__ __forceinline__ int stat_slot(int q) {
  const int slot[kTileStats] = {ST_CHECKS, ST_EVALUATED, ST_CULLED, ST_FALLBACK_ROWS,
                                ST_PENALTY_FAILS, ST_BATCH_FAILS, ST_BATCH_SIZE};
  return slot[q];
}

// Sums of the per-tile counters into the stats slots (one atomic per
// workgroup and counter).
template <int N>
__global__ __launch_bounds__(256) void k_tile_stats(const unsigned long long* __restrict__ ts,
                                                    long long npairs, int tiles,
                                                    const long long* __restrict__ npairs_dev,
                                                    unsigned long long* __restrict__ stats) {
  __shared__ unsigned long long red[N];
  if (threadIdx.x < N) red[threadIdx.x] = 0;
  __syncthreads();
  const long long ntiles = (npairs_dev && *npairs_dev < npairs ? *npairs_dev : npairs) * tiles;
  unsigned long long acc[N] = {};
  for (long long t = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; t < ntiles;
       t += static_cast<long long>(gridDim.x) * 256)
    for (int q = 0; q < N; ++q) acc[q] += ts[t * N + q];
  for (int q = 0; q < N; ++q) {
    unsigned long long v = acc[q];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(&red[q], v);
  }
  __syncthreads();
  if (threadIdx.x < N && red[threadIdx.x])
    atomicAdd(&stats[stat_slot(threadIdx.x)], red[threadIdx.x]);
}

// The tail of a captured detection over at most kTailPairs pairs, in one
// workgroup in place of three launches: the tile counters' sums (as
// k_tile_stats), the per-pair contact counts (as k_tile_sums; with one tile
// per pair the detection wrote them directly) and their exclusive prefix
// sums with the total at offs[npairs] (as scan_counts).
constexpr int kTailPairs = 4096;

template <int N>
__global__ __launch_bounds__(1024) void k_detect_tail_small(
    const unsigned long long* __restrict__ ts, const long long* __restrict__ npairs_dev,
    unsigned long long* __restrict__ stats, const int* __restrict__ tile_count, int tiles,
    int npairs, int* __restrict__ counts, long long* __restrict__ offs) {
  __shared__ unsigned long long red[N];
  __shared__ long long s_wave[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (t < N) red[t] = 0;
  __syncthreads();
  const long long ntiles =
      (npairs_dev && *npairs_dev < npairs ? *npairs_dev : static_cast<long long>(npairs)) * tiles;
  unsigned long long acc[N] = {};
  for (long long k = t; k < ntiles; k += 1024)
    for (int q = 0; q < N; ++q) acc[q] += ts[k * N + q];
  for (int q = 0; q < N; ++q) {
    unsigned long long v = acc[q];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0 && v) atomicAdd(&red[q], v);
  }
  // four consecutive pairs per thread
  int c[4];
  long long local = 0;
  for (int u = 0; u < 4; ++u) {
    const int k = 4 * t + u;
    int v = 0;
    if (k < npairs) {
      if (tiles > 1) {
        for (int q = 0; q < tiles; ++q) v += tile_count[static_cast<long long>(k) * tiles + q];
        counts[k] = v;
      } else {
        v = counts[k];
      }
    }
    c[u] = v;
    local += v;
  }
  long long incl = local;
  for (int o = 1; o < 64; o <<= 1) {
    const long long u = __shfl_up(incl, o);
    incl += lane >= o ? u : 0;
  }
  if (lane == 63) s_wave[w] = incl;
  __syncthreads();
  long long before = 0;
  for (int q = 0; q < w; ++q) before += s_wave[q];
  long long run = before + incl - local;
  for (int u = 0; u < 4; ++u) {
    const int k = 4 * t + u;
    if (k < npairs) offs[k] = run;
    run += c[u];
  }
  if (t == 1023) offs[npairs] = before + incl;
  if (t < N && red[t]) atomicAdd(&stats[stat_slot(t)], red[t]);
}

// GJK over the particles' vertex replicas (gjk.cpp:25-100 with the core of
// gjk.cpp:418-460), one wave per particle pair: the support searches are
// lane-parallel (first index of the strict extremum after a wave
// reduction); the simplex arithmetic is uniform across the wave.  At most one
// contact per pair, when |P-Q| <= epsA + epsB; triA = triB = -1.
__device__ __forceinline__ int wave_extremum(double bd, int bi, bool maximal) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double od = __shfl_xor(bd, o);
    const int oi = __shfl_xor(bi, o);
    const bool better = oi >= 0 && (bi < 0 || (maximal ? od > bd : od < bd) ||
                                    (od == bd && oi < bi));
    bd = better ? od : bd;
    bi = better ? oi : bi;
  }
  return bi;
}

__global__ __launch_bounds__(256) void k_gjk(DetectArgs g) {
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= g.npairs) return;
  unsigned long long* ts = g.tile_stats + static_cast<long long>(k) * g.nstats;
  if (g.npairs_dev && k >= *g.npairs_dev) {
    if (lane == 0) g.tile_count[k] = 0;
    if (lane < g.nstats) ts[lane] = 0;
    return;
  }
  const Pair p = load_pair(g, k);
  const int na = 3 * p.nA, nb = 3 * p.nB, ba = 3 * p.oA, bb = 3 * p.oB;
  auto pa = [&](int i) { return V3<double>{g.x[ba + i], g.y[ba + i], g.z[ba + i]}; };
  auto pb = [&](int i) { return V3<double>{g.x[bb + i], g.y[bb + i], g.z[bb + i]}; };
  auto min_a = [&](const double* v) {
    double bd = 1.7976931348623157e308;
    int bi = -1;
    for (int i = lane; i < na; i += 64) {
      const double c[3] = {g.x[ba + i], g.y[ba + i], g.z[ba + i]};
      const double d = gdot(c, v);
      if (d < bd) {
        bd = d;
        bi = i;
      }
    }
    return wave_extremum(bd, bi, false);
  };
  auto max_b = [&](const double* v) {
    double bd = -1.7976931348623157e308;
    int bi = -1;
    for (int i = lane; i < nb; i += 64) {
      const double c[3] = {g.x[bb + i], g.y[bb + i], g.z[bb + i]};
      const double d = gdot(c, v);
      if (d > bd) {
        bd = d;
        bi = i;
      }
    }
    return wave_extremum(bd, bi, true);
  };
  double P[3] = {0, 0, 0}, Q[3] = {0, 0, 0};
  bool ok = na > 0 && nb > 0;
  if (ok) gjk_core(na, nb, pa, pb, min_a, max_b, P, Q, &ok);
  const V3<double> vP = {P[0], P[1], P[2]}, vQ = {Q[0], Q[1], Q[2]};
  const bool emit = ok && pq_dist(vP, vQ) <= p.margin;
  if (lane == 0) {
    if (emit) {
      const unsigned long long slot = atomicAdd(g.counter, 1ull);
      if (static_cast<long long>(slot) < g.cap) {
        dh_contact c;
        make_contact(p, k, -1, -1, vP, vQ, &c);
        c.pad_ = 0;
        g.temp[slot] = c;
      }
    }
    g.tile_count[k] = emit ? 1 : 0;
  }
  if (lane < kTileStats) {
    ts[lane] = lane == TS_CHECKS ? static_cast<unsigned long long>(p.nA) * p.nB
             : lane == TS_EVALUATED ? 1ull : 0ull;
  }
}

// exclusive scan of per-pair counts (two levels, 1024 per block)
// live (may be null): the scan covers the first min(n, *live) entries only.
__device__ __forceinline__ int scan_len(int n, const unsigned long long* live) {
  return live && *live < static_cast<unsigned long long>(n) ? static_cast<int>(*live) : n;
}

__global__ __launch_bounds__(1024) void k_scan_blocks(const int* __restrict__ in, int n,
                                                      long long* __restrict__ out,
                                                      long long* __restrict__ block_sums,
                                                      const unsigned long long* __restrict__ live) {
  __shared__ long long buf[1024];
  n = scan_len(n, live);
  if (static_cast<long long>(blockIdx.x) * 1024 >= n) {  // past the live entries
    if (threadIdx.x == 0) block_sums[blockIdx.x] = 0;
    return;
  }
  const int i = blockIdx.x * 1024 + threadIdx.x;
  const long long v = (i < n) ? in[i] : 0;
  buf[threadIdx.x] = v;
  __syncthreads();
  for (int s = 1; s < 1024; s <<= 1) {
    const long long t = (threadIdx.x >= s) ? buf[threadIdx.x - s] : 0;
    __syncthreads();
    buf[threadIdx.x] += t;
    __syncthreads();
  }
  if (i < n) out[i] = buf[threadIdx.x] - v;
  if (threadIdx.x == 1023) block_sums[blockIdx.x] = buf[1023];
}

// The whole scan in one workgroup when n <= 1,024 (the small scenes' pair
// and particle counts): offs[0..n) exclusive, offs[n] the total.
__global__ __launch_bounds__(1024) void k_scan_single(const int* __restrict__ in, int n,
                                                      long long* __restrict__ out,
                                                      const unsigned long long* __restrict__ live) {
  __shared__ long long buf[1024];
  n = scan_len(n, live);
  const int i = threadIdx.x;
  const long long v = i < n ? in[i] : 0;
  buf[i] = v;
  __syncthreads();
  for (int s = 1; s < 1024; s <<= 1) {
    const long long t = i >= s ? buf[i - s] : 0;
    __syncthreads();
    buf[i] += t;
    __syncthreads();
  }
  if (i < n) out[i] = buf[i] - v;
  if (i == 1023) out[n] = buf[1023];
}

// Exclusive scan of the block sums in place, by one workgroup: 1,024 at a
// time with a running carry.
__global__ __launch_bounds__(1024) void k_scan_sums(long long* __restrict__ sums, int nb) {
  __shared__ long long buf[1024];
  __shared__ long long carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nb; base += 1024) {
    const int i = base + threadIdx.x;
    const long long v = i < nb ? sums[i] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int s = 1; s < 1024; s <<= 1) {
      const long long t = (threadIdx.x >= s) ? buf[threadIdx.x - s] : 0;
      __syncthreads();
      buf[threadIdx.x] += t;
      __syncthreads();
    }
    const long long c = carry;
    if (i < nb) sums[i] = c + buf[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = c + buf[1023];
    __syncthreads();
  }
}

// Adds the block offsets; the last element's thread also writes the total
// out[n] (out[0] = 0 when n = 0).
__global__ __launch_bounds__(1024) void k_scan_add(long long* __restrict__ out, int n,
                                                   const long long* __restrict__ sums,
                                                   const int* __restrict__ in,
                                                   const unsigned long long* __restrict__ live) {
  n = scan_len(n, live);
  const int i = blockIdx.x * 1024 + threadIdx.x;
  if (i < n) {
    const long long o = out[i] + sums[blockIdx.x];
    out[i] = o;
    if (i == n - 1) out[n] = o + in[i];
  } else if (n == 0 && i == 0) {
    out[0] = 0;
  }
}

// k_scan_add for at most 1,024 blocks, without the block-sum scan: each
// block first adds up the raw sums of the blocks before it.
__global__ __launch_bounds__(1024) void k_scan_add_prefix(long long* __restrict__ out, int n,
                                                          const long long* __restrict__ sums,
                                                          const int* __restrict__ in,
                                                          const unsigned long long* __restrict__ live) {
  __shared__ long long part[16];
  n = scan_len(n, live);
  const int b = blockIdx.x, tid = threadIdx.x;
  if (static_cast<long long>(b) * 1024 >= n && !(n == 0 && b == 0)) return;
  long long v = tid < b ? sums[tid] : 0;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if ((tid & 63) == 0) part[tid >> 6] = v;
  __syncthreads();
  long long base = 0;
  for (int w = 0; w < 16; ++w) base += part[w];
  const int i = b * 1024 + tid;
  if (i < n) {
    const long long o = out[i] + base;
    out[i] = o;
    if (i == n - 1) out[n] = o + in[i];
  } else if (n == 0 && i == 0) {
    out[0] = 0;
  }
}

// Per-pair contact counts from the per-tile counts.
__global__ __launch_bounds__(256) void k_tile_sums(const int* __restrict__ tile_count, int tiles,
                                                   int npairs, int* __restrict__ counts) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= npairs) return;
  int c = 0;
  for (int t = 0; t < tiles; ++t) c += tile_count[static_cast<long long>(k) * tiles + t];
  counts[k] = c;
}

// Contacts into pair order: pair offset + the counts of the pair's earlier
// tiles + the rank within the tile.
__global__ __launch_bounds__(256) void k_scatter(const dh_contact* __restrict__ temp, long long n,
                                                 const long long* __restrict__ offs,
                                                 const int* __restrict__ tile_count, int tiles,
                                                 dh_contact* __restrict__ out,
                                                 const unsigned long long* __restrict__ n_dev,
                                                 Report report) {
  // n is the capacity (of temp and out), the count is read from n_dev
  const long long live = static_cast<long long>(*n_dev) < n ? static_cast<long long>(*n_dev) : n;
  for (long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; i < live;
       i += static_cast<long long>(gridDim.x) * 256) {
    dh_contact c = temp[i];
    const int pair = c.pair / tiles;
    long long dst = offs[pair] + c.pad_;
    for (int t = pair * tiles; t < c.pair; ++t) dst += tile_count[t];
    if (dst >= n) continue;  // more contacts than the capacity (reported by the caller)
    c.pair = pair;
    c.pad_ = 0;
    out[dst] = c;
  }
  if (blockIdx.x == 0) report_write(report, threadIdx.x, 256);
}

// Survivor queue, pass 2: every wave takes one segment of k_detect_wave's through
// the plane test, the edge-pair axes (and, when tuned on, the binary32 screen)
// and bfSolver.  What a test leaves waits in a list in LDS until 64 entries
// are there, so that each stage runs with every lane busy although the one
// before it drops most.  The entries stay in order, so the contacts of an item
// come out in row-major order and their rank is a running count, and the
// records of a segment follow each other without a counter that all waves
// share.  Bound by vector issue: 152 us for the hopper's 1.78e6 entries and
// 644,000 contacts (a lane per entry, with its scan, reservation and unordered
// contacts: 250 us); four waves per SIMD would spill (166 us).
struct QueueLists {
  int a[128], b[128];  // entries for the axes, for bfSolver
};

// Lanes' places in a wave's list of n entries; the whole wave calls it.
__device__ __forceinline__ int list_append(int* list, int n, bool keep, int e) {
  const unsigned long long m = __ballot(keep);
  if (keep) list[n + lane_prefix(m)] = e;
  wave_lds_fence();
  return n + __popcll(m);
}

// The first 64 entries of a list of n off it: the lane's entry (-1 past the
// end); the rest move to the front.
__device__ __forceinline__ int list_take(int* list, int& n, int lane) {
  const int e = lane < n ? list[lane] : -1;
  const int rest = n > 64 ? n - 64 : 0;
  const int r = lane < rest ? list[64 + lane] : 0;
  wave_lds_fence();
  if (lane < rest) list[lane] = r;
  wave_lds_fence();
  n = rest;
  return e;
}

__device__ __forceinline__ double entry_margin(const DetectArgs& g, const int4& en) {
  const int k = en.x / g.tiles;
  return g.eps[g.pairs[2 * k]] + g.eps[g.pairs[2 * k + 1]];
}

// Ranks of the emitting lanes within their items (runs of one item, in order)
// after `carry` contacts of item `carry_item` so far; the last lane of each
// run writes the item's count.  The whole wave calls it.
__device__ __forceinline__ int item_rank(const DetectArgs& g, bool emit, int item, int lane,
                                         int& carry_item, int& carry) {
  const unsigned long long mask = __ballot(emit), below = (1ull << lane) - 1;
  if (!mask) return 0;
  const unsigned long long before = mask & below;
  const int prev = before ? 63 - __clzll(static_cast<long long>(before)) : lane;
  const int prev_item = __shfl(item, prev);  // by every lane: prev must take part
  const bool head = emit && (!before || prev_item != item);
  const unsigned long long heads = __ballot(head);
  const unsigned long long upto = heads & (below | 1ull << lane);
  const int first = upto ? 63 - __clzll(static_cast<long long>(upto)) : lane;
  int rank = __popcll(before & ~((1ull << first) - 1));
  if (item == carry_item && first == __builtin_ctzll(mask)) rank += carry;
  const int last = 63 - __clzll(static_cast<long long>(mask));
  const unsigned long long after = mask & ~(below | 1ull << lane);
  const bool tail = emit && (!after || (heads >> __builtin_ctzll(after) & 1));
  if (tail) g.tile_count[item] = rank + 1;
  carry_item = __shfl(item, last);
  carry = __shfl(rank, last) + 1;
  return rank;
}

// The n entries at q through the tests and bfSolver; their contacts' records
// to rec, in order.  Returns the number of records, and the first and the last
// item that has one with their counts.  With kFilter the entries that the tests
// leave are compacted in place instead, and counted.
struct StreamEnds {
  int n, first, nfirst, last, nlast;
};

template <bool SCREEN, bool kFilter>
__device__ __forceinline__ StreamEnds solve_stream(const DetectArgs& g, int4* __restrict__ q, int n,
                                                   QueueRecord* __restrict__ rec, QueueLists& L,
                                                   int lane) {
  int na = 0, nb = 0, base = 0, out = 0, carry_item = -1, carry = 0;
  int first = -1, nfirst = 0;
  for (;;) {
    const bool eof = base >= n;
    if (nb >= 64 || (eof && na == 0 && nb > 0)) {
      const int e = list_take(L.b, nb, lane);
      int4 en = make_int4(-1, 0, 0, 0);
      if (e >= 0) en = q[e];
      if (kFilter) {
        // every entry before these has been read: the places are free
        const unsigned long long m = __ballot(e >= 0);
        if (e >= 0) q[out + lane_prefix(m)] = en;
        out += __popcll(m);
        continue;
      }
      bool emit = false;
      V3<double> P = {0, 0, 0}, Q = {0, 0, 0};
      if (e >= 0) {
        bf_solver(load_tri(g, en.y), load_tri(g, en.z), P, Q);
        emit = pq_dist(P, Q) <= entry_margin(g, en);
      }
      const int rank = item_rank(g, emit, en.x, lane, carry_item, carry);
      const unsigned long long m = __ballot(emit);
      if (emit) {
        QueueRecord r;
        r.item = en.x;
        r.tris = en.w;
        r.rank = rank;
        r.pad_ = 0;
        r.pq[0] = P.x; r.pq[1] = P.y; r.pq[2] = P.z;
        r.pq[3] = Q.x; r.pq[4] = Q.y; r.pq[5] = Q.z;
        rec[out + lane_prefix(m)] = r;
      }
      if (m && out == 0) first = __shfl(en.x, __builtin_ctzll(m));
      nfirst += __popcll(__ballot(emit && en.x == first));
      out += __popcll(m);
    } else if (na >= 64 || (eof && na > 0)) {
      const int e = list_take(L.a, na, lane);
      bool keep = false;
      if (e >= 0) {
        const int4 en = q[e];
        const Tri<double> A = load_tri(g, en.y), B = load_tri(g, en.z);
        const double margin = entry_margin(g, en);
        keep = !edge_axes_apart(A, B, axis_reach(A, B, margin)) &&
               !(SCREEN && screened_far(A, B, margin));
      }
      nb = list_append(L.b, nb, keep, e);
    } else if (!eof) {
      const int e = base + lane;
      bool keep = false;
      if (e < n) {
        const int4 en = q[e];
        keep = !plane_apart(load_tri(g, en.y), load_tri(g, en.z), entry_margin(g, en));
      }
      na = list_append(L.a, na, keep, e);
      base += 64;
    } else {
      break;
    }
  }
  return {out, first, nfirst, carry_item, carry};
}

// The part of a heavy segment's n entries that each of a workgroup's waves
// takes, in whole rounds of 64.
__device__ __forceinline__ int segment_part(int n) { return (n + 255) / 256 * 64; }

// A wave per segment; then the workgroup's four waves share each of its segments
// with more than g.heavy entries, so that one pair of particles in deep
// contact does not keep a single wave at work (the funnel's heaviest pairs
// have 400 contacts: 100 us without, 69 us with).  An item that goes on from
// one part of a segment to the next has the later part's ranks raised by the
// contacts before (applied in k_queue_write).
template <bool SCREEN, bool kFilter>
__global__ __launch_bounds__(256, 3) void k_queue_solve(DetectArgs g) {
  __shared__ QueueLists lists[4];
  __shared__ StreamEnds ends[4];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  // the workgroup's segments: four of the waves' own, then of the pool's.  They
  // lie far apart: neighbours hold neighbouring pairs, which are heavy together
  const int grid = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
  const int most = 4 + (g.shape.segments() - g.shape.regions + grid - 1) / grid;
  auto number = [&](int i) { return i < 4 ? i * grid + b : g.shape.regions + (i - 4) * grid + b; };
  auto count = [&](int i) {
    const int r = number(i);
    return i < most && r < (i < 4 ? g.shape.regions : g.shape.segments()) ? g.rcount[r] : 0;
  };
  for (int i0 = 0; i0 < most; i0 += 64) {  // 64 of them at a time
    unsigned long long light, heavy;       // the wave's; the same in all waves
    int known = 0;  // entries of the first, 0 afterwards (read again)
    {
      const int entries = count(i0 + lane);
      light = __ballot(entries > 0 && entries <= g.heavy && (lane & 3) == w);
      heavy = __ballot(entries > g.heavy);
      if (light) known = __builtin_amdgcn_readlane(entries, __builtin_ctzll(light));
    }
    while (light | heavy) {
      const bool shared = light == 0;
      const int l = __builtin_ctzll(shared ? heavy : light);
      if (shared) heavy &= heavy - 1;
      else light &= light - 1;
      const int r = number(i0 + l), total = known ? known : g.rcount[r];
      known = 0;
      int begin = 0, n = total;
      if (shared) {
        const int part = segment_part(total);
        begin = w * part < total ? w * part : total;
        n = total - begin < part ? total - begin : part;
      }
      const long long at = g.shape.place(r) + begin;
      const StreamEnds e = solve_stream<SCREEN, kFilter>(g, g.queue + at, n, g.rec + at, lists[w], lane);
      if (!shared) {
        if (lane == 0) g.rcount[(kFilter ? 0 : g.shape.segments()) + r] = e.n;
        continue;
      }
      if (lane == 0) ends[w] = e;
      __syncthreads();
      if (threadIdx.x == 0) {
        int item = -1, count = 0;
        for (int q = 0; q < 4; ++q) {
          const StreamEnds s = ends[q];
          const int base = s.n > 0 && s.first == item ? count : 0;
          int* c = g.rparts + 8 * static_cast<long long>(r) + 2 * q;
          c[0] = s.n;
          c[1] = base;
          if (s.n == 0) continue;
          if (base > 0) g.tile_count[s.first] = base + s.nfirst;
          count = s.first == s.last ? base + s.nfirst : s.nlast;
          item = s.last;
        }
      }
      __syncthreads();
    }
  }
}

// The records of entries that another kernel has solved and left in the
// records' places by entry (`rank` of those that emit is not 0), moved to the
// front in order.
__global__ __launch_bounds__(256) void k_queue_record(DetectArgs g) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + static_cast<int>(threadIdx.x >> 6);
  if (r >= g.shape.segments()) return;
  const long long at = g.shape.place(r);
  const int n = g.rcount[r];
  int out = 0, carry_item = -1, carry = 0;
  for (int base = 0; base < n; base += 64) {
    const long long e = at + base + lane;
    const bool emit = base + lane < n && g.rec[e].rank != 0;
    int4 en = make_int4(-1, 0, 0, 0);
    double pq[6] = {};
    if (emit) {
      en = g.queue[e];
#pragma unroll
      for (int c = 0; c < 6; ++c) pq[c] = g.rec[e].pq[c];
    }
    const int rank = item_rank(g, emit, en.x, lane, carry_item, carry);
    const unsigned long long m = __ballot(emit);
    if (emit) {  // every record up to here has been read: the places are free
      QueueRecord q;
      q.item = en.x;
      q.tris = en.w;
      q.rank = rank;
      q.pad_ = 0;
#pragma unroll
      for (int c = 0; c < 6; ++c) q.pq[c] = pq[c];
      g.rec[at + out + lane_prefix(m)] = q;
    }
    out += __popcll(m);
  }
  if (lane == 0) g.rcount[g.shape.segments() + r] = out;
}

// Pass 3, after the pairs' offsets: the records' contacts, each at its place,
// and those that the full kernel left in `temp` (*in_temp of them).  A
// workgroup per segment: a record waits for a chain of loads, which a wave per
// segment went through once per 64 records (hopper of 15,651 spheres 51 us,
// 46 us now, near the copy rate).
__device__ __forceinline__ long long contact_place(const DetectArgs& g, int item, int rank,
                                                   const long long* __restrict__ offs) {
  const int k = item / g.tiles;
  long long dst = offs[k] + rank;
  for (int t = k * g.tiles; t < item; ++t) dst += g.tile_count[t];
  return dst;
}

__global__ __launch_bounds__(256) void k_queue_write(DetectArgs g, const long long* __restrict__ offs,
                                                     dh_contact* __restrict__ out, long long cap,
                                                     const unsigned long long* __restrict__ in_temp,
                                                     unsigned long long* __restrict__ found,
                                                     Report report) {
  const int r = blockIdx.x;
  const int total = g.rcount[r];
  const bool heavy = total > g.heavy;
  for (int p = 0; p < (heavy ? 4 : total > 0 ? 1 : 0); ++p) {
    const int* c = g.rparts + 8 * static_cast<long long>(r) + 2 * p;
    const int n = heavy ? c[0] : g.rcount[g.shape.segments() + r];
    if (n == 0) continue;
    const QueueRecord* rec =
        g.rec + g.shape.place(r) + (heavy ? p * segment_part(total) : 0);
    const int base = heavy ? c[1] : 0, first = rec[0].item;
    for (int e = threadIdx.x; e < n; e += 256) {
      const QueueRecord q = rec[e];
      const long long dst = contact_place(g, q.item, q.rank + (q.item == first ? base : 0), offs);
      if (dst >= cap) continue;  // past the capacity: dropped (reported by the caller)
      const int k = q.item / g.tiles;
      const unsigned tris = static_cast<unsigned>(q.tris);
      dh_contact ct;
      make_contact(load_pair(g, k), k, static_cast<int>(tris & 0xffffu),
                   static_cast<int>(tris >> 16), V3<double>{q.pq[0], q.pq[1], q.pq[2]},
                   V3<double>{q.pq[3], q.pq[4], q.pq[5]}, &ct);
      ct.pad_ = 0;
      out[dst] = ct;
    }
  }
  const unsigned long long nt = *in_temp < static_cast<unsigned long long>(g.cap)
                                    ? *in_temp : static_cast<unsigned long long>(g.cap);
  for (unsigned long long i = blockIdx.x * 256ull + threadIdx.x; i < nt; i += gridDim.x * 256ull) {
    dh_contact c = g.temp[i];
    const long long dst = contact_place(g, c.pair, c.pad_, offs);
    if (dst >= cap) continue;
    c.pair /= g.tiles;
    c.pad_ = 0;
    out[dst] = c;
  }
  if (found && blockIdx.x == 0 && threadIdx.x == 0)
    *found = static_cast<unsigned long long>(
        offs[g.npairs_dev && *g.npairs_dev < g.npairs ? *g.npairs_dev : g.npairs]);
  if (blockIdx.x == 0) report_write(report, threadIdx.x, 256);
}

int queue_learned(const int4* queue, const int* pairs, int tiles, const QueueShape& shape,
                  const int* rcount, const double* x, const double* y, const double* z,
                  const double* eps, int* flags, int flag_stride, double* pq, int pq_stride,
                  hipStream_t st);
int queue_learned_reserve(long long n);

struct DetectScratch {
  DevBuf temp, counter, stats, error, counts, offs, sums, tiles, tstats, iskip, tmax;
  DevBuf queue, qrec, qcounts, rparts, deferred, wlist, found;
};
static DetectScratch g_scratch;

// The largest triangle count of a particle, per geometry (tri_offset, n,
// ntri): k_chunk_cull runs only on scenes with particles of more than
// kRowBlock triangles.  A stale entry changes the speed, never the result
// (the pre-pass is exact, and without it detect_item does the same tests).
struct TriMax {
  const int* tri_offset = nullptr;
  int n = -1, ntri = -1, max_tris = 0;
};
static TriMax g_trimax;

__global__ __launch_bounds__(256) void k_max_tris(const int* __restrict__ off, int n,
                                                  int* __restrict__ out) {
  int m = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    m = max(m, off[i + 1] - off[i]);
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
  if ((threadIdx.x & 63) == 0 && m > 0) atomicMax(out, m);
}

// With sync, computes and caches a geometry not cached (one read-back);
// without (inside a capture), answers 0 for it.
static int particle_max_tris(const dh_geometry* g, hipStream_t st, bool sync) {
  if (g_trimax.tri_offset == g->tri_offset && g_trimax.n == g->nparticles &&
      g_trimax.ntri == g->ntri_total)
    return g_trimax.max_tris;
  if (!sync || g->nparticles <= 0) return 0;
  if (g_scratch.tmax.grow(sizeof(int))) return 0;
  int m = 0;
  if (hipMemsetAsync(g_scratch.tmax.ptr, 0, sizeof(int), st) != hipSuccess) return 0;
  const unsigned grid = grid_for(g->nparticles, 256) < 1024 ? grid_for(g->nparticles, 256) : 1024;
  hipLaunchKernelGGL(k_max_tris, grid, 256, 0, st, g->tri_offset, g->nparticles,
                     g_scratch.tmax.as<int>());
  if (hipMemcpyAsync(&m, g_scratch.tmax.ptr, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return 0;
  g_trimax = {g->tri_offset, g->nparticles, g->ntri_total, m};
  return m;
}

// Before a capture of a step on this geometry: fills the cache above.
int detect_prepare(const dh_geometry* geom, hipStream_t st) {
  particle_max_tris(geom, st, true);
  return DH_OK;
}

// Scratch of scan_counts for up to n entries (before a capture).
int scan_reserve(int n) {
  const int nb = (n + 1023) / 1024 > 0 ? (n + 1023) / 1024 : 1;
  return g_scratch.sums.grow(sizeof(long long) * (nb + 1));
}

// Exclusive scan of counts[0..m) into offs[0..m), offs[m] the total, where
// m = n, or min(n, *live) when live is given (read when the kernels run);
// `sums` holds scan_sums_len(n) block sums (unused when n <= 1,024).
static int scan_counts_upto(const int* counts, int n, const unsigned long long* live,
                            long long* offs, long long* sums, hipStream_t st) {
  if (n <= 1024) {
    hipLaunchKernelGGL(k_scan_single, 1, 1024, 0, st, counts, n, offs, live);
    DH_HIP_CHECK(hipGetLastError());
    return DH_OK;
  }
  const int nb = (n + 1023) / 1024;
  hipLaunchKernelGGL(k_scan_blocks, nb, 1024, 0, st, counts, n, offs, sums, live);
  if (nb <= 1024) {  // two launches: the add pass sums the block sums before it
    hipLaunchKernelGGL(k_scan_add_prefix, nb, 1024, 0, st, offs, n, sums, counts, live);
  } else {
    hipLaunchKernelGGL(k_scan_sums, 1, 1024, 0, st, sums, nb);
    hipLaunchKernelGGL(k_scan_add, nb, 1024, 0, st, offs, n, sums, counts, live);
  }
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

// offs[0..n]: exclusive prefix sums of counts, offs[n] = total.
int scan_counts_with(const int* counts, int n, long long* offs, long long* sums,
                     hipStream_t st) {
  return scan_counts_upto(counts, n, nullptr, offs, sums, st);
}

int scan_sums_len(int n) { return (n + 1023) / 1024 > 0 ? (n + 1023) / 1024 + 1 : 2; }

// The same with the library's own block-sum scratch.
int scan_counts(const int* counts, int n, long long* offs, hipStream_t st) {
  if (n > 1024) {
    int rc = g_scratch.sums.grow(sizeof(long long) * scan_sums_len(n));
    if (rc) return rc;
  }
  return scan_counts_with(counts, n, offs, g_scratch.sums.as<long long>(), st);
}

// Workgroups of a detection launch over `items`: one per item, or the
// persistent grid of detect_wg_per_cu workgroups per CU.
static unsigned detect_grid(long long items) {
  const int per_cu = tuning().detect_wg_per_cu;
  long long g = items;
  if (per_cu > 0 && g > static_cast<long long>(device_cus()) * per_cu)
    g = static_cast<long long>(device_cus()) * per_cu;
  return static_cast<unsigned>(g < 1 ? 1 : g);
}

template <int M>
static void launch_detect(unsigned items, size_t shm, hipStream_t st, const DetectArgs& a) {
  if (M == DH_BF && a.item_skip) {
    const long long wg = (static_cast<long long>(items) + 3) / 4;
    const long long cap = static_cast<long long>(device_cus()) * 32;
    hipLaunchKernelGGL(k_chunk_cull, static_cast<unsigned>(wg < cap ? (wg > 0 ? wg : 1) : cap),
                       256, 0, st, a, static_cast<int>(items),
                       const_cast<unsigned char*>(a.item_skip));
  }
  hipLaunchKernelGGL(k_detect<M>, detect_grid(items), 256, shm, st, a,
                     static_cast<int>(items));
}

static void launch_tile_stats(const DetectArgs& a, hipStream_t st) {
  const long long ntiles = static_cast<long long>(a.npairs) * a.tiles;
  if (ntiles <= 0) return;
  long long grid = (ntiles + 255) / 256;
  if (grid > 256) grid = 256;
  const auto f = a.nstats == kBfStats ? k_tile_stats<kBfStats> : k_tile_stats<kTileStats>;
  hipLaunchKernelGGL(f, static_cast<unsigned>(grid), 256, 0, st, a.tile_stats,
                     static_cast<long long>(a.npairs), a.tiles, a.npairs_dev, a.stats);
}

// Row ranges per particle pair: enough workgroups to fill the 256 CUs
// several times over when the pairs are few (detect_tile_target workgroups
// in all, at most detect_max_tiles per pair), one per pair otherwise.
static int tiles_for(long long npairs, int method) {
  if (method == DH_GJK || npairs <= 0) return 1;
  const long long target = tuning().detect_tile_target, cap = tuning().detect_max_tiles;
  long long t = (target + npairs - 1) / npairs;
  return static_cast<int>(t < 1 ? 1 : (t > cap ? cap : t));
}

// Entries of the survivor queue for `items` items and `cap` contacts: 16 per item
// and 65,536, or 2.5 per contact where that is more (packings leave 2.1 to 2.9
// survivors per contact), the latter up to 2^24.  What does not fit is deferred.
static long long queue_total(long long items, long long cap) {
  const long long by_items = 16 * items + 65536, contacts = cap < 1ll << 24 ? cap : 1ll << 24;
  const long long by_contacts = 5 * contacts / 2 < 1ll << 24 ? 5 * contacts / 2 : 1ll << 24;
  const long long n = by_items > by_contacts ? by_items : by_contacts;
  return n < 1ll << 28 ? n : 1ll << 28;
}

// The queue's shape: half of the entries are the waves' own segments (as many
// waves as the CUs hold at once), of at least 1,024 each (335 MB), the other
// half the pool; with 16 items per wave and more, which makes the segments
// alike, three quarters and one.  (Own segments of 512 or 256 entries: funnel
// fill's step 2 and 3 % slower, as a wave whose items go on in the pool waits
// for it.)  Of segments that are not alike, those with more than 256 entries are
// shared by four waves in k_queue_solve.  An item may queue up to 2,048 entries,
// 1,024 where one wave alone takes a segment through the learned decision
// (1,024 always: captured packing of 512 at half its pitch 977 us, 931 so).
struct QueuePlan {
  unsigned groups;
  QueueShape shape;
  int heavy, most;
};

static QueuePlan queue_plan(long long items, long long total, bool learned) {
  QueuePlan q;
  const long long wg = (items + kWavesPerGroup - 1) / kWavesPerGroup;
  const long long waves = static_cast<long long>(device_cus()) * 8;
  q.groups = static_cast<unsigned>(wg < 1 ? 1 : (wg < waves ? wg : waves));
  q.shape.regions = static_cast<int>(q.groups) * kWavesPerGroup;
  const bool alike = items >= 16ll * q.shape.regions;
  const long long pool = alike ? total / 4 : total / 2;
  const long long own = (total - pool) / q.shape.regions / 64 * 64;
  q.shape.rcap = static_cast<int>(own < 1024 ? 1024 : own);
  const long long block = (pool / 8192 + 63) / 64 * 64;
  q.shape.block = static_cast<int>(block < 1024 ? 1024 : block);
  const long long blocks = pool / q.shape.block / kPoolParts;
  q.shape.blocks = static_cast<int>(blocks < 1 ? 1 : blocks);
  q.heavy = learned || alike ? 0x7fffffff : 256;
  q.most = learned ? 1024 : 2048;
  return q;
}

// Places of the queue path's counters in g_scratch.qcounts: the lists' lengths,
// the pool's parts, then the segments' entries and contacts.
enum QueueCount : int {
  QC_WLIST = 0, QC_DEFERRED, QC_NEXT, QC_POOL,
  QC_SEGMENTS = QC_POOL + kPoolParts * kPoolStride
};

static int queue_counts(const QueuePlan& q) { return QC_SEGMENTS + 2 * q.shape.segments(); }

// Buffers of the queue path (before a capture).
static int queue_reserve(const QueuePlan& q, long long items, bool learned) {
  int rc;
  if ((rc = g_scratch.queue.grow(sizeof(int4) * q.shape.entries()))) return rc;
  if ((rc = g_scratch.qrec.grow(sizeof(QueueRecord) * q.shape.entries()))) return rc;
  if ((rc = g_scratch.qcounts.grow(sizeof(unsigned) * queue_counts(q)))) return rc;
  if ((rc = g_scratch.rparts.grow(sizeof(int) * 8 * q.shape.segments()))) return rc;
  if ((rc = g_scratch.deferred.grow(sizeof(int) * (items + 1)))) return rc;
  if ((rc = g_scratch.wlist.grow(sizeof(WaveItem) * (items + 1)))) return rc;
  if ((rc = g_scratch.found.grow(sizeof(unsigned long long)))) return rc;
  return learned ? queue_learned_reserve(q.shape.entries()) : DH_OK;
}

static void queue_bind(DetectArgs& a, const QueuePlan& q) {
  unsigned* c = g_scratch.qcounts.as<unsigned>();
  a.queue = g_scratch.queue.as<int4>();
  a.shape = q.shape;
  a.most = q.most;
  a.pool = c + QC_POOL;
  a.rcount = reinterpret_cast<int*>(c + QC_SEGMENTS);
  a.rparts = g_scratch.rparts.as<int>();
  a.heavy = q.heavy;
  a.rec = g_scratch.qrec.as<QueueRecord>();
  a.deferred = g_scratch.deferred.as<int>();
  a.ndeferred = c + QC_DEFERRED;
  a.wlist = g_scratch.wlist.as<WaveItem>();
  a.nwlist = c + QC_WLIST;
}

// A DH_BF detection through the survivor queue: the mid-phase, the items it
// could not queue in full (as many as *ndeferred), then the queue's solve.
// Every launch is for the capacity and reads the live lengths, so nothing is
// read back on the way.
static int queue_detect(const DetectArgs& a, const QueuePlan& q, unsigned items, bool learned,
                        hipStream_t st) {
  const unsigned cus = static_cast<unsigned>(device_cus());
  const int group = items <= kFewItems ? 256 : 1024;
  hipLaunchKernelGGL(k_lane_cull, items > 0 ? grid_for(items, group) : 1u, group, 0, st, a,
                     static_cast<int>(items));
  hipLaunchKernelGGL(k_detect_wave, q.groups, 64 * kWavesPerGroup, 0, st, a);
  DetectArgs f = a;
  f.item_list = a.deferred;
  f.nitems_dev = a.ndeferred;
  f.item_next = g_scratch.qcounts.as<unsigned>() + QC_NEXT;
  // usually none to do: a grid for the capacity would cost a dispatch per item
  hipLaunchKernelGGL(k_detect<DH_BF>, items < 4 * cus ? items : 4 * cus, 256, 0, st, f,
                     static_cast<int>(items));
  const auto solve = learned ? (a.fp32_screen ? k_queue_solve<true, true> : k_queue_solve<false, true>)
                             : (a.fp32_screen ? k_queue_solve<true, false> : k_queue_solve<false, false>);
  hipLaunchKernelGGL(solve, grid_for(q.shape.regions, 4), 256, 0, st, a);
  if (learned) {
    int rc;
    static_assert(sizeof(QueueRecord) == 64, "a record's strides below");
    if ((rc = queue_learned(a.queue, a.pairs, a.tiles, a.shape, a.rcount, a.x, a.y, a.z, a.eps,
                            &a.rec->rank, 16, a.rec->pq, 8, st)))
      return rc;
    hipLaunchKernelGGL(k_queue_record, grid_for(q.shape.segments(), 4), 256, 0, st, a);
  }
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

// The DetectArgs of a call without its queue.
static DetectArgs detect_args(const dh_geometry* geom, const int* pairs, int npairs,
                              const long long* np_dev, long long cap, int tiles, int* tile_count,
                              bool bf, const double* pbox, const double* bbox,
                              const double* psph) {
  DetectArgs a = {};
  a.x = geom->x;
  a.y = geom->y;
  a.z = geom->z;
  a.tri_offset = geom->tri_offset;
  a.eps = geom->eps;
  a.friction = geom->friction;
  a.id = geom->id;
  a.pairs = pairs;
  a.npairs = npairs;
  a.temp = g_scratch.temp.as<dh_contact>();
  a.cap = cap;
  a.counter = g_scratch.counter.as<unsigned long long>();
  a.tiles = tiles;
  a.tile_count = tile_count;
  a.nstats = bf ? kBfStats : kTileStats;
  a.tile_stats = g_scratch.tstats.as<unsigned long long>();
  a.stats = g_scratch.stats.as<unsigned long long>();
  a.error = g_scratch.error.as<int>();
  a.npairs_dev = np_dev;
  a.pbox = pbox;
  a.psph = pbox ? psph : nullptr;
  a.bbox = bbox;
  a.fp32_screen = tuning().detect_fp32_screen;
  return a;
}

// After the detection: the tile counters summed, the pairs' contact counts and
// their offsets (of the live pairs).
static int pair_offsets(const DetectArgs& a, int* counts, long long* offs, hipStream_t st) {
  if (a.npairs <= kTailPairs) {
    const auto f = a.nstats == kBfStats ? k_detect_tail_small<kBfStats>
                                        : k_detect_tail_small<kTileStats>;
    hipLaunchKernelGGL(f, 1, 1024, 0, st, a.tile_stats, a.npairs_dev, a.stats, a.tile_count,
                       a.tiles, a.npairs, counts, offs);
    DH_HIP_CHECK(hipGetLastError());
    return DH_OK;
  }
  launch_tile_stats(a, st);
  if (a.tiles > 1)
    hipLaunchKernelGGL(k_tile_sums, grid_for(a.npairs, 256), 256, 0, st, a.tile_count, a.tiles,
                       a.npairs, counts);
  int rc = g_scratch.sums.grow(sizeof(long long) * scan_sums_len(a.npairs));
  if (rc) return rc;
  return scan_counts_upto(counts, a.npairs,
                          reinterpret_cast<const unsigned long long*>(a.npairs_dev), offs,
                          g_scratch.sums.as<long long>(), st);
}

// At least min_tiles tiles per pair.
static int detect_pairs_tiled(int method, const dh_geometry* geom, const int* pairs, int npairs,
                              int min_tiles, dh_contact* out, long long cap, long long* n_total,
                              int* pair_count_user, long long* offs_out, dh_stats* stats,
                              hipStream_t st, const double* pbox, const double* bbox,
                              const double* psph) {
  int rc;
  // DH_BF_LEARNED: DH_BF with the survivor queue always on, its pairs
  // through the learned decision
  const bool learned = method == DH_BF_LEARNED;
  if (learned) method = DH_BF;
  const long long temp_cap = cap > 0 ? cap : 1;
  if ((rc = g_scratch.temp.grow(sizeof(dh_contact) * temp_cap))) return rc;
  if ((rc = g_scratch.counter.grow(sizeof(unsigned long long)))) return rc;
  if ((rc = g_scratch.stats.grow(sizeof(unsigned long long) * ST_COUNT))) return rc;
  if ((rc = g_scratch.error.grow(sizeof(int)))) return rc;
  if ((rc = g_scratch.counts.grow(sizeof(int) * (npairs + 1)))) return rc;
  if ((rc = g_scratch.offs.grow(sizeof(long long) * (npairs + 1)))) return rc;
  int* counts = pair_count_user ? pair_count_user : g_scratch.counts.as<int>();
  int tiles = tiles_for(npairs, method);
  if (tiles < min_tiles && method != DH_GJK) tiles = min_tiles;
  int* tile_count = counts;
  if (tiles > 1) {
    if ((rc = g_scratch.tiles.grow(sizeof(int) * static_cast<size_t>(npairs) * tiles))) return rc;
    tile_count = g_scratch.tiles.as<int>();
  }
  const long long nitems = static_cast<long long>(npairs) * tiles;
  const bool bf = method == DH_BF;
  if ((rc = g_scratch.tstats.grow(sizeof(unsigned long long) * (bf ? kBfStats : kTileStats) *
                                  nitems)))
    return rc;
  DetectArgs a = detect_args(geom, pairs, npairs, nullptr, cap, tiles, tile_count, bf, pbox, bbox,
                             psph);
  // the queue costs launches: for many items only
  const bool queued =
      bf && (learned || queue_items(static_cast<long long>(npairs) * tiles_for(npairs, method),
                                    geom->ntri_total, geom->nparticles) >=
                            tuning().detect_queue_min_items);
  QueuePlan plan = {};
  if (queued) {
    // a shorter queue where the memory does not allow this one
    for (long long total = queue_total(nitems, cap);; total /= 2) {
      plan = queue_plan(nitems, total, learned);
      if (!(rc = queue_reserve(plan, nitems, learned))) break;
      if (total <= 65536) return rc;
      (void)hipGetLastError();
    }
    queue_bind(a, plan);
  }
  zero_async(ZeroRegions{{g_scratch.counter.as<unsigned>(), g_scratch.stats.as<unsigned>(),
                          g_scratch.error.as<unsigned>(),
                          queued ? g_scratch.qcounts.as<unsigned>() : nullptr},
                         {2, 2 * ST_COUNT, 1, queued ? queue_counts(plan) : 0}},
             st);
  const size_t shm_rows = 2 * kMaxRowTriangles * sizeof(int) + 8 + kMaxRowTriangles * 8;
  const unsigned items = static_cast<unsigned>(nitems);
  if (bf && !queued && pbox && bbox &&
      particle_max_tris(geom, st, true) > kRowBlock) {
    if ((rc = g_scratch.iskip.grow(items > 0 ? items : 1))) return rc;
    a.item_skip = g_scratch.iskip.as<unsigned char>();
  }
  switch (method) {
    case DH_BF:
      if (!queued) launch_detect<DH_BF>(items, 0, st, a);
      else if ((rc = queue_detect(a, plan, items, learned, st))) return rc;
      break;
    case DH_PENALTY: launch_detect<DH_PENALTY>(items, 0, st, a); break;
    case DH_PENALTY_STAT: launch_detect<DH_PENALTY_STAT>(items, 0, st, a); break;
    case DH_HYBRID_BATCH: launch_detect<DH_HYBRID_BATCH>(items, shm_rows, st, a); break;
    case DH_HYBRID_TRIANGLE: launch_detect<DH_HYBRID_TRIANGLE>(items, shm_rows, st, a); break;
    case DH_HYBRID_BATCH_STAT: launch_detect<DH_HYBRID_BATCH_STAT>(items, shm_rows, st, a); break;
    case DH_HYBRID_TRIANGLE_STAT:
      launch_detect<DH_HYBRID_TRIANGLE_STAT>(items, shm_rows, st, a);
      break;
    case DH_GJK:
      hipLaunchKernelGGL(k_gjk, (items + 3) / 4, 256, 0, st, a);
      break;
    default:
      return set_error(DH_ERR_UNSUPPORTED, "dh_detect_pairs: method %d", method);
  }
  DH_HIP_CHECK(hipGetLastError());
  long long* offs = offs_out ? offs_out : g_scratch.offs.as<long long>();
  if ((rc = pair_offsets(a, counts, offs, st))) return rc;
  // the contacts to their places, with the counts reported: one wait for all
  Report report;
  if ((rc = report_open(report))) return rc;
  report_add(report, offs + npairs, 2);
  report_add(report, g_scratch.error.ptr, 1);
  report_add(report, g_scratch.stats.ptr, 2 * ST_COUNT);
  if (queued) {
    hipLaunchKernelGGL(k_queue_write, static_cast<unsigned>(plan.shape.segments()), 256, 0, st, a, offs,
                       out, cap, a.counter, nullptr, report);
  } else {
    const long long wg = (cap + 255) / 256;
    hipLaunchKernelGGL(k_scatter, static_cast<unsigned>(wg < 1 ? 1 : (wg < 2048 ? wg : 2048)), 256,
                       0, st, a.temp, cap, offs, tile_count, tiles, out, a.counter, report);
  }
  if ((rc = report_wait(st))) return rc;
  unsigned long long total;
  int err;
  unsigned long long st_host[ST_COUNT];
  std::memcpy(&total, report.mail, sizeof(total));
  std::memcpy(&err, report.mail + 2, sizeof(err));
  std::memcpy(st_host, report.mail + 3, sizeof(st_host));
  if (err == DE_REF_UB)
    return set_error(DH_ERR_REF_UB,
                     "hybridWithPerTriangleFallBack reads row iA < nTriB of A: nTriB > nTriA is "
                     "out of bounds in the reference (hybrid.cpp:130)");
  if (err == DE_TOO_LONG)
    return set_error(DH_ERR_ARG, "more than %d triangles in a particle (reference row limit)",
                     kMaxRowTriangles);
  *n_total = static_cast<long long>(total);
  if (stats) {
    for (int i = 0; i < 17; ++i) stats->newton_histogram[i] += st_host[ST_HIST + i];
    stats->penalty_fails += st_host[ST_PENALTY_FAILS];
    stats->batch_fails += st_host[ST_BATCH_FAILS];
    stats->batch_size += st_host[ST_BATCH_SIZE];
    stats->triangle_checks += st_host[ST_CHECKS];
    stats->pairs_evaluated += st_host[ST_EVALUATED];
    stats->fallback_rows += st_host[ST_FALLBACK_ROWS];
    stats->pairs_culled += st_host[ST_CULLED];
  }
  if (static_cast<long long>(total) > cap) return DH_ERR_CAPACITY;
  return DH_OK;
}

int detect_pairs_impl(int method, const dh_geometry* geom, const int* pairs, int npairs,
                      dh_contact* out, long long cap, long long* n_total, int* pair_count_user,
                      long long* offs_out, dh_stats* stats, hipStream_t st,
                      const double* pbox, const double* bbox, const double* psph) {
  return detect_pairs_tiled(method, geom, pairs, npairs, 1, out, cap, n_total, pair_count_user,
                            offs_out, stats, st, pbox, bbox, psph);
}

int detect_reserve(const dh_geometry* geom, int pair_cap, long long contact_cap, int method);

// Tiles of the captured step, sized for half the pair capacity live.
static int graph_tiles(int pair_cap) { return tiles_for(pair_cap / 2 > 0 ? pair_cap / 2 : 1, DH_BF); }

// Whether a captured step's detection goes through the survivor queue.
static bool graph_queued(int method, const dh_geometry* geom, int pair_cap) {
  const long long items = static_cast<long long>(pair_cap) * graph_tiles(pair_cap);
  return method == DH_BF_LEARNED ||
         (method == DH_BF && queue_items(items, geom->ntri_total, geom->nparticles) >=
                                 tuning().detect_queue_min_items);
}

// Detection for a captured step: launches for `pair_cap` pairs of which
// *np_dev are live, contacts into `out` (capacity contact_cap), per-pair
// counts and offsets; no host synchronisation.  Counters stay on the device:
// dev_counters()[0] = contacts found (may exceed contact_cap), error flag.
int detect_pairs_graph(int method, const dh_geometry* geom, const int* pairs, int pair_cap,
                       const long long* np_dev, dh_contact* out, long long contact_cap,
                       int* counts, long long* offs, hipStream_t st, const double* pbox,
                       const double* bbox, const double* psph) {
  int rc;
  if ((rc = detect_reserve(geom, pair_cap, contact_cap, method))) return rc;
  const bool learned = method == DH_BF_LEARNED;
  const bool queued = graph_queued(method, geom, pair_cap);
  if (learned) method = DH_BF;
  const int tiles = graph_tiles(pair_cap);
  const unsigned items = static_cast<unsigned>(static_cast<long long>(pair_cap) * tiles);
  const QueuePlan plan =
      queued ? queue_plan(items, queue_total(items, contact_cap), learned) : QueuePlan{};
  zero_async(ZeroRegions{{g_scratch.counter.as<unsigned>(), g_scratch.stats.as<unsigned>(),
                          g_scratch.error.as<unsigned>(),
                          queued ? g_scratch.qcounts.as<unsigned>() : nullptr},
                         {2, 2 * ST_COUNT, 1, queued ? queue_counts(plan) : 0}},
             st);
  const bool bf = method == DH_BF;
  DetectArgs a = detect_args(geom, pairs, pair_cap, np_dev, contact_cap, tiles,
                             tiles > 1 ? g_scratch.tiles.as<int>() : counts, bf, pbox, bbox, psph);
  // the chunk pre-pass on the geometries detect_prepare found walls in
  if (bf && !queued && pbox && bbox && particle_max_tris(geom, st, false) > kRowBlock)
    a.item_skip = g_scratch.iskip.as<unsigned char>();
  if (queued) queue_bind(a, plan);
  switch (method) {
    case DH_BF:
      if (!queued) launch_detect<DH_BF>(items, 0, st, a);
      else if ((rc = queue_detect(a, plan, items, learned, st))) return rc;
      break;
    case DH_PENALTY: launch_detect<DH_PENALTY>(items, 0, st, a); break;
    default:
      return set_error(DH_ERR_UNSUPPORTED, "captured step: method %d (use DH_BF or DH_PENALTY)",
                       method);
  }
  if ((rc = pair_offsets(a, counts, offs, st))) return rc;
  if (queued) {
    hipLaunchKernelGGL(k_queue_write, static_cast<unsigned>(plan.shape.segments()), 256, 0, st, a, offs,
                       out, contact_cap, a.counter, g_scratch.found.as<unsigned long long>(), Report{});
  } else {
    const long long wg = (contact_cap + 255) / 256;
    hipLaunchKernelGGL(k_scatter, static_cast<unsigned>(wg < 2048 ? wg : 2048), 256, 0, st, a.temp,
                       contact_cap, offs, a.tile_count, tiles, out, a.counter, Report{});
  }
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

// Buffers of detect_pairs_graph (call before a capture: no allocation may
// happen inside one).
int detect_reserve(const dh_geometry* geom, int pair_cap, long long contact_cap, int method) {
  int rc;
  if (graph_queued(method, geom, pair_cap)) {
    const long long items = static_cast<long long>(pair_cap) * graph_tiles(pair_cap);
    const bool learned = method == DH_BF_LEARNED;
    const QueuePlan plan = queue_plan(items, queue_total(items, contact_cap), learned);
    if ((rc = queue_reserve(plan, items, learned))) return rc;
  }
  if ((rc = g_scratch.temp.grow(sizeof(dh_contact) * (contact_cap > 0 ? contact_cap : 1)))) return rc;
  if ((rc = g_scratch.counter.grow(sizeof(unsigned long long)))) return rc;
  if ((rc = g_scratch.stats.grow(sizeof(unsigned long long) * ST_COUNT))) return rc;
  if ((rc = g_scratch.error.grow(sizeof(int)))) return rc;
  if ((rc = g_scratch.sums.grow(sizeof(long long) * scan_sums_len(pair_cap)))) return rc;
  const int tiles = graph_tiles(pair_cap);
  if (tiles > 1 &&
      (rc = g_scratch.tiles.grow(sizeof(int) * static_cast<size_t>(pair_cap) * tiles)))
    return rc;
  if (method == DH_BF &&
      (rc = g_scratch.iskip.grow(static_cast<size_t>(pair_cap) * tiles + 1)))
    return rc;
  if ((rc = g_scratch.tstats.grow(sizeof(unsigned long long) * kTileStats *
                                  static_cast<size_t>(pair_cap) * tiles)))
    return rc;
  return DH_OK;
}

// Device addresses of the detection counters of a captured step: the contacts
// found, the error flag and the statistics.
const unsigned long long* detect_counter_dev(int method, const dh_geometry* geom,
                                             int pair_cap) {
  return graph_queued(method, geom, pair_cap) ? g_scratch.found.as<unsigned long long>()
                                        : g_scratch.counter.as<unsigned long long>();
}
const int* detect_error_dev() { return g_scratch.error.as<int>(); }
const unsigned long long* detect_stats_dev() { return g_scratch.stats.as<unsigned long long>(); }

// Particles and contacts of a host call that go through pinned memory, which is
// kept (65,536 contacts take 9.4 MB, 233,000 triangles 16); more are copied.
constexpr size_t kPinnedBytes = 16u << 20;

__global__ __launch_bounds__(256) void k_fetch(const double* __restrict__ src,
                                               double* __restrict__ dst, long long n) {
  for (long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<long long>(gridDim.x) * 256)
    dst[i] = src[i];
}

// _batchError of the *Stat drivers: maxErr added once per row, in row order
// and pair order (hybrid.cpp:240,530).
static double batch_error_sum(double acc, double max_err, int rows) {
  for (int r = 0; r < rows; ++r) acc += max_err;
  return acc;
}

}  // namespace dh

using namespace dh;

extern "C" {

int dh_exclusive_scan(const int* counts_dev, int n, int64_t* offs_dev, void* stream) {
  int rc = ensure_init();
  if (rc) return rc;
  if (n < 0 || !offs_dev || (n > 0 && !counts_dev))
    return set_error(DH_ERR_ARG, "dh_exclusive_scan: bad arguments");
  return scan_counts(counts_dev, n, reinterpret_cast<long long*>(offs_dev), as_stream(stream));
}

int dh_detect_pairs(int method, const dh_geometry* geom, const int* pairs_dev, int npairs,
                    dh_contact* out_dev, int cap, int* n_out, int* pair_count_dev,
                    dh_stats* stats, void* stream) {
  int rc = ensure_init();
  if (rc) return rc;
  if (!geom || !n_out || npairs < 0 || cap < 0 || (npairs > 0 && !pairs_dev))
    return set_error(DH_ERR_ARG, "dh_detect_pairs: bad arguments");
  *n_out = 0;
  if (npairs == 0) return DH_OK;
  long long total = 0;
  rc = detect_pairs_impl(method, geom, pairs_dev, npairs, out_dev, cap, &total, pair_count_dev,
                         nullptr, stats, as_stream(stream), nullptr, nullptr, nullptr);
  *n_out = static_cast<int>(total);
  if (stats && (method == DH_HYBRID_BATCH_STAT || method == DH_HYBRID_TRIANGLE_STAT) &&
      (rc == DH_OK || rc == DH_ERR_CAPACITY)) {
    // sequential _batchError accumulation needs eps and row counts per pair
    std::vector<int> pr(2 * static_cast<size_t>(npairs));
    std::vector<int> off(geom->nparticles + 1);
    std::vector<double> eps(geom->nparticles);
    DH_HIP_CHECK(hipMemcpy(pr.data(), pairs_dev, sizeof(int) * pr.size(), hipMemcpyDeviceToHost));
    DH_HIP_CHECK(hipMemcpy(off.data(), geom->tri_offset, sizeof(int) * off.size(),
                           hipMemcpyDeviceToHost));
    DH_HIP_CHECK(hipMemcpy(eps.data(), geom->eps, sizeof(double) * eps.size(),
                           hipMemcpyDeviceToHost));
    double acc = stats->batch_error;
    for (int k = 0; k < npairs; ++k) {
      const int a = pr[2 * k], b = pr[2 * k + 1];
      acc = batch_error_sum(acc, (eps[a] + eps[b]) / 16, off[a + 1] - off[a]);
      (void)b;
    }
    stats->batch_error = acc;
  }
  return rc;
}

int dh_detect_pair(int method, const double* xA, const double* yA, const double* zA, int nTriA,
                   double epsA, int frictionA, int idA, const double* xB, const double* yB,
                   const double* zB, int nTriB, double epsB, int frictionB, int idB,
                   dh_contact* out, int cap, int* n_out, dh_stats* stats) {
  int rc = ensure_init();
  if (rc) return rc;
  if (!n_out || nTriA < 0 || nTriB < 0 || cap < 0 || (cap > 0 && !out))
    return set_error(DH_ERR_ARG, "dh_detect_pair: bad arguments");
  *n_out = 0;
  if (method == DH_HYBRID_TRIANGLE && nTriB > nTriA)
    return set_error(DH_ERR_REF_UB,
                     "hybridWithPerTriangleFallBack reads row iA < nTriB of A: nTriB > nTriA is "
                     "out of bounds in the reference (hybrid.cpp:130)");
  if (nTriA == 0 || nTriB == 0) return DH_OK;
  // The two particles go to the device in one block, up to kPinnedBytes staged
  // in pinned memory and fetched from there by a kernel, and the contacts come
  // back into pinned memory, written by the kernel that orders them: one wait per
  // call (seven copies in and one out cost 170 of the 205 us of a 20 x 20 call).
  struct Meta {
    double eps[2];
    int off[3];
    int fric[2];
    int id[2];
    int pairs[2];
    int pad_[3];
  };
  static_assert(sizeof(Meta) % 16 == 0, "the vertices follow on a 16-byte boundary");
  static DevBuf geo, outbuf;
  static PinnedBuf stage, pinned_out;
  const size_t na = 3 * static_cast<size_t>(nTriA), nb = 3 * static_cast<size_t>(nTriB);
  const size_t nv = na + nb, block = sizeof(Meta) + 3 * nv * sizeof(double);
  if ((rc = geo.grow(block))) return rc;
  const Meta m = {{epsA, epsB},   {0, nTriA, nTriA + nTriB}, {frictionA ? 1 : 0, frictionB ? 1 : 0},
                  {idA, idB},     {0, 1},                    {0, 0, 0}};
  const double* axes[3][2] = {{xA, xB}, {yA, yB}, {zA, zB}};
  const bool staged = block <= kPinnedBytes;
  if (staged && (rc = stage.grow(block))) return rc;
  char* to = staged ? static_cast<char*>(stage.ptr) : geo.as<char>();
  // to the pinned block, or to the device (which waits for earlier calls' work)
  auto put = [&](size_t at, const void* from, size_t bytes) -> int {
    if (staged)
      std::memcpy(to + at, from, bytes);
    else
      DH_HIP_CHECK(hipMemcpy(to + at, from, bytes, hipMemcpyHostToDevice));
    return DH_OK;
  };
  if ((rc = put(0, &m, sizeof(m)))) return rc;
  for (int q = 0; q < 3; ++q) {
    const size_t at = sizeof(Meta) + q * nv * sizeof(double);
    if ((rc = put(at, axes[q][0], na * sizeof(double)))) return rc;
    if ((rc = put(at + na * sizeof(double), axes[q][1], nb * sizeof(double)))) return rc;
  }
  if (staged) {
    const long long words = static_cast<long long>(block / 8);
    hipLaunchKernelGGL(k_fetch, grid_for(words, 256) < 256 ? grid_for(words, 256) : 256, 256, 0,
                       nullptr, static_cast<const double*>(stage.ptr), geo.as<double>(), words);
    DH_HIP_CHECK(hipGetLastError());
  }
  const Meta* dm = geo.as<Meta>();
  dh_geometry g;
  g.x = reinterpret_cast<double*>(geo.as<char>() + sizeof(Meta));
  g.y = g.x + nv;
  g.z = g.y + nv;
  g.tri_offset = dm->off;
  g.eps = dm->eps;
  g.friction = dm->fric;
  g.id = dm->id;
  g.nparticles = 2;
  g.ntri_total = nTriA + nTriB;
  const long long dcap = cap > 0 ? cap : 1;
  const size_t out_bytes = sizeof(dh_contact) * dcap;
  const bool direct = out_bytes <= kPinnedBytes;
  if ((rc = direct ? pinned_out.grow(out_bytes) : outbuf.grow(out_bytes))) return rc;
  dh_contact* dev_out = direct ? static_cast<dh_contact*>(pinned_out.ptr) : outbuf.as<dh_contact>();
  // Tiles of 256 triangle pairs, one per thread, where each is solved, and of
  // 4,096 where most are culled, up to the 64 of the largest
  // detect_max_tiles: 16 tiles left 320 x 80 triangles to 16 CUs (hybrid
  // kernel 69 us, 37 us with 64).
  const long long per = method == DH_BF || method == DH_BF_LEARNED ? 4096 : 256;
  const long long want = static_cast<long long>(nTriA) * nTriB / per;
  long long total = 0;
  rc = detect_pairs_tiled(method, &g, dm->pairs, 1, static_cast<int>(want < 64 ? want : 64),
                          dev_out, cap, &total, nullptr, nullptr, stats, nullptr, nullptr, nullptr,
                          nullptr);
  *n_out = static_cast<int>(total);
  if (rc != DH_OK) return rc;
  if (stats && (method == DH_HYBRID_BATCH_STAT || method == DH_HYBRID_TRIANGLE_STAT))
    stats->batch_error = batch_error_sum(stats->batch_error, (epsA + epsB) / 16, nTriA);
  if (total > 0 && direct)
    std::memcpy(out, dev_out, sizeof(dh_contact) * total);
  else if (total > 0)
    DH_HIP_CHECK(hipMemcpy(out, dev_out, sizeof(dh_contact) * total, hipMemcpyDeviceToHost));
  return DH_OK;
}

}  // extern "C"
