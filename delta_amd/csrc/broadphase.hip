// broadphase.hip — candidate particle pairs from a uniform hash grid.
//
// The reference has no broad phase on its engine path (Engine.cpp:272-295 is
// an O(N^2) loop with an optional bounding-sphere test; Peano supplies a grid
// in the app).  Here the candidate set is defined exactly: every pair (i<j),
// not both obstacles, whose particle AABBs inflated by their margins (plus a
// 0.5e-9 m band each) overlap.  The grid is a search structure only: cell
// size >= the largest inflated extent of a non-obstacle particle guarantees
// that overlapping boxes sit in neighbouring cells, so the grid result equals
// the all-pairs test.  "Large" particles -- obstacles (floors, funnels, boxes)
// and any particle whose inflated box outgrows the cell, which the reference's
// non-orthogonal rotation update (dynamics.cpp:78) can cause -- are kept out
// of the grid and tested against every particle.  Output pairs are sorted (i ascending, then
// j ascending) regardless of hash-bucket order.
#include <mutex>
#include <vector>

#include "runtime.hpp"

namespace dh {

struct Aabb {
  double lo[3], hi[3];
};

// Pairs of vertex replicas per lane that the box pass loads at once and keeps
// for the sphere pass (a particle of up to 128 * kAabbHeld replicas is read
// once).
constexpr int kAabbHeld = 4;
constexpr int kAabbWaves = 8;  // particles per workgroup

// Two consecutive doubles, loaded as 16 bytes from any 8-byte boundary (a
// particle's replicas start at one).
struct alignas(8) Two {
  double a, b;
};

// The vertices [0, nv) from v0 in blocks of 128 * kAabbHeld, a lane's two at a
// time; NaN past the end (min, max and the sphere skip NaN).
struct HeldVertices {
  Two x[kAabbHeld], y[kAabbHeld], z[kAabbHeld];

  __device__ __forceinline__ void load(const double* __restrict__ px,
                                       const double* __restrict__ py,
                                       const double* __restrict__ pz, int v0, int b, int nv,
                                       int lane) {
#pragma unroll
    for (int k = 0; k < kAabbHeld; ++k) {
      const int v = b + 128 * k + 2 * lane;
      x[k] = y[k] = z[k] = Two{NAN, NAN};
      if (v + 1 < nv) {
        x[k] = *reinterpret_cast<const Two*>(px + v0 + v);
        y[k] = *reinterpret_cast<const Two*>(py + v0 + v);
        z[k] = *reinterpret_cast<const Two*>(pz + v0 + v);
      } else if (v < nv) {
        x[k].a = px[v0 + v];
        y[k].a = py[v0 + v];
        z[k].a = pz[v0 + v];
      }
    }
  }
  __device__ __forceinline__ double far2(const double c[3]) const {
    double r2 = 0.0;
#pragma unroll
    for (int k = 0; k < kAabbHeld; ++k) {
      double dx = x[k].a - c[0], dy = y[k].a - c[1], dz = z[k].a - c[2];
      r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
      dx = x[k].b - c[0], dy = y[k].b - c[1], dz = z[k].b - c[2];
      r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
    }
    return r2;
  }
};

// v of the lane that `ctrl` (a DPP control) names, which is in the same row of 16.
template <int ctrl>
__device__ __forceinline__ double row_move(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// The smallest over each row of 16 lanes, in all of them, without LDS: lanes
// xor 1, xor 2, then the row's halves and the row mirrored.
__device__ __forceinline__ double row_min(double v) {
  v = fmin(v, row_move<0xb1>(v));
  v = fmin(v, row_move<0x4e>(v));
  v = fmin(v, row_move<0x141>(v));
  return fmin(v, row_move<0x140>(v));
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

__device__ __forceinline__ double wave_min(double v) {
  v = row_min(v);
  return fmin(fmin(lane_value(v, 0), lane_value(v, 16)),
              fmin(lane_value(v, 32), lane_value(v, 48)));
}

// The box of the wave's lanes' boxes, in all lanes.  A first exchange leaves
// lo in the lower and -hi in the upper 32 lanes, so that one reduction does
// for both.
__device__ __forceinline__ void wave_box(double lo[3], double hi[3]) {
  const bool upper = __lane_id() >= 32;
  for (int q = 0; q < 3; ++q) {
    const double up = -hi[q];
    const double other = __shfl_xor(upper ? lo[q] : up, 32);
    const double v = row_min(fmin(upper ? up : lo[q], other));
    lo[q] = fmin(lane_value(v, 0), lane_value(v, 16));
    hi[q] = -fmin(lane_value(v, 32), lane_value(v, 48));
  }
}

__device__ __forceinline__ void store_box(Aabb* __restrict__ box, const double* __restrict__ eps,
                                          int i, const double lo[3], const double hi[3]) {
  const double m = eps[i] + 0.5e-9;
  Aabb bx;
  for (int q = 0; q < 3; ++q) {
    bx.lo[q] = lo[q] - m;
    bx.hi[q] = hi[q] + m;
  }
  box[i] = bx;
}

__device__ __forceinline__ void store_sphere(double* __restrict__ sph, int i, const double c[3],
                                             double r2) {
  sph[4 * i] = c[0];
  sph[4 * i + 1] = c[1];
  sph[4 * i + 2] = c[2];
  sph[4 * i + 3] = sqrt(r2);
}

// A particle's box (inflated by its margin), its chunks' boxes when it has
// more triangles than one row block (chunk c of 64 triangles at
// cbox[t0 / 64 + i + c], an index that grows with i and c, so no two chunks
// share it) and, with sph, a bounding sphere: the vertex box's centre and the
// largest vertex distance from it (NaN coordinates drop out, as from the box).
// A wave per particle, its replicas read once; the workgroup's waves share a
// particle with chunks (one wave took 51 us for a 2,048-triangle funnel, the
// longest chain of the scene's pass: 23 us now).  HBM bound: the 1.5 GB of the
// 2e5-particle box take 287 us (5.2 TB/s; 304 us with reductions through LDS
// shuffles and 8-byte loads, 348 us where all workgroups wait for the one
// particle that they share).
__global__ __launch_bounds__(64 * kAabbWaves) void k_particle_aabb(
    int n, const double* __restrict__ x, const double* __restrict__ y,
    const double* __restrict__ z, const int* __restrict__ tri_offset,
    const double* __restrict__ eps, Aabb* __restrict__ box, Aabb* __restrict__ cbox,
    double* __restrict__ sph) {
  __shared__ double red[kAabbWaves][7];
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  {
    const int i = blockIdx.x * kAabbWaves + w;
    const int t0 = i < n ? tri_offset[i] : 0, t1 = i < n ? tri_offset[i + 1] : 0;
    const bool chunked = cbox && t1 - t0 > kRowBlock;
    const int v0 = 3 * t0, nv = t1 > t0 ? 3 * (t1 - t0) : 0;
    if (i < n && !chunked) {
      double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
      HeldVertices h;
      for (int b = 0; b < nv; b += 128 * kAabbHeld) {
        h.load(x, y, z, v0, b, nv, lane);
#pragma unroll
        for (int k = 0; k < kAabbHeld; ++k) {
          lo[0] = fmin(fmin(lo[0], h.x[k].a), h.x[k].b);
          lo[1] = fmin(fmin(lo[1], h.y[k].a), h.y[k].b);
          lo[2] = fmin(fmin(lo[2], h.z[k].a), h.z[k].b);
          hi[0] = fmax(fmax(hi[0], h.x[k].a), h.x[k].b);
          hi[1] = fmax(fmax(hi[1], h.y[k].a), h.y[k].b);
          hi[2] = fmax(fmax(hi[2], h.z[k].a), h.z[k].b);
        }
      }
      wave_box(lo, hi);
      if (lane == 0) store_box(box, eps, i, lo, hi);
      if (sph) {
        const double c[3] = {0.5 * (lo[0] + hi[0]), 0.5 * (lo[1] + hi[1]), 0.5 * (lo[2] + hi[2])};
        double r2 = 0.0;
        // the replicas come from registers when one block held them all
        for (int b = 0; b < nv; b += 128 * kAabbHeld) {
          if (nv > 128 * kAabbHeld) h.load(x, y, z, v0, b, nv, lane);
          r2 = fmax(r2, h.far2(c));
        }
        r2 = -wave_min(-r2);
        if (lane == 0) store_sphere(sph, i, c, r2);
      }
    }
  }
  if (!cbox) return;
  for (int p = 0; p < kAabbWaves; ++p) {
    const int i = blockIdx.x * kAabbWaves + p;
    if (i >= n) break;
    const int t0 = tri_offset[i], t1 = tri_offset[i + 1];
    if (t1 - t0 <= kRowBlock) continue;  // the same for the whole workgroup
    const int v0 = 3 * t0, nv = 3 * (t1 - t0);
    double plo[3] = {INFINITY, INFINITY, INFINITY}, phi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int c = w; 64 * c < t1 - t0; c += kAabbWaves) {
      const int b0 = 64 * c, b1 = b0 + 64 < t1 - t0 ? b0 + 64 : t1 - t0;
      double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int v = 3 * b0 + 64 * k + lane;
        const bool in = v < 3 * b1;
        const double cx = in ? x[v0 + v] : NAN, cy = in ? y[v0 + v] : NAN,
                     cz = in ? z[v0 + v] : NAN;
        lo[0] = fmin(lo[0], cx);
        lo[1] = fmin(lo[1], cy);
        lo[2] = fmin(lo[2], cz);
        hi[0] = fmax(hi[0], cx);
        hi[1] = fmax(hi[1], cy);
        hi[2] = fmax(hi[2], cz);
      }
      wave_box(lo, hi);
      if (lane == 0) {
        Aabb bx;
        for (int q = 0; q < 3; ++q) {
          bx.lo[q] = lo[q];
          bx.hi[q] = hi[q];
        }
        cbox[t0 / 64 + i + c] = bx;
      }
      for (int q = 0; q < 3; ++q) {
        plo[q] = fmin(plo[q], lo[q]);
        phi[q] = fmax(phi[q], hi[q]);
      }
    }
    if (lane == 0)
      for (int q = 0; q < 3; ++q) {
        red[w][q] = plo[q];
        red[w][3 + q] = phi[q];
      }
    __syncthreads();
    for (int o = 0; o < kAabbWaves; ++o)
      for (int q = 0; q < 3; ++q) {
        plo[q] = fmin(plo[q], red[o][q]);
        phi[q] = fmax(phi[q], red[o][3 + q]);
      }
    if (threadIdx.x == 0) store_box(box, eps, i, plo, phi);
    if (sph) {
      const double c[3] = {0.5 * (plo[0] + phi[0]), 0.5 * (plo[1] + phi[1]),
                           0.5 * (plo[2] + phi[2])};
      double r2 = 0.0;
      for (int b = 128 * kAabbHeld * w; b < nv; b += 128 * kAabbHeld * kAabbWaves) {
        HeldVertices h;
        h.load(x, y, z, v0, b, nv, lane);
        r2 = fmax(r2, h.far2(c));
      }
      r2 = -wave_min(-r2);
      if (lane == 0) red[w][6] = r2;
      __syncthreads();
      for (int o = 0; o < kAabbWaves; ++o) r2 = fmax(r2, red[o][6]);
      if (threadIdx.x == 0) store_sphere(sph, i, c, r2);
    }
    __syncthreads();  // the next particle reuses the reductions
  }
}

static void launch_aabb(const dh_geometry* g, Aabb* box, Aabb* cbox, double* sph, hipStream_t st) {
  hipLaunchKernelGGL(k_particle_aabb, grid_for(g->nparticles, kAabbWaves), 64 * kAabbWaves, 0, st,
                     g->nparticles, g->x, g->y, g->z, g->tri_offset, g->eps, box, cbox, sph);
}

__device__ __forceinline__ bool overlap(const Aabb& a, const Aabb& b) {
  for (int q = 0; q < 3; ++q)
    if (a.lo[q] > b.hi[q] || b.lo[q] > a.hi[q]) return false;
  return true;
}

__device__ __forceinline__ void cell_of(const Aabb& b, double inv_h, long long c[3]) {
  for (int q = 0; q < 3; ++q) c[q] = static_cast<long long>(floor(0.5 * (b.lo[q] + b.hi[q]) * inv_h));
}

__device__ __forceinline__ unsigned hash_cell(long long cx, long long cy, long long cz,
                                              unsigned mask) {
  unsigned long long h = static_cast<unsigned long long>(cx) * 0x9E3779B97F4A7C15ull ^
                         static_cast<unsigned long long>(cy) * 0xC2B2AE3D27D4EB4Full ^
                         static_cast<unsigned long long>(cz) * 0x165667B19E3779F9ull;
  h ^= h >> 29;
  return static_cast<unsigned>(h) & mask;
}

// The grid is a cell list sorted by hash bucket: bucket b holds the
// particles entry[cstart[b] .. cstart[b+1]) (a counting sort: counts,
// exclusive scan, scatter), so a bucket is one contiguous range and its
// members load without pointer chasing.
//
// A member is found with its box and cell beside its number, so that a search
// waits for one load per round (with the number first and the box after it,
// and 64-bit cells formed again for every candidate, the 2e5-particle box took
// 198 us; 123 us now).  Cells are compared in their low 32 bits: two that agree there and
// differ are 2^32 cells apart and their boxes do not overlap.
struct alignas(64) GridEntry {
  Aabb box;
  int cell[3];
  int id;
};

struct GridArgs {
  const Aabb* box;
  const int* obstacle;  // may be null
  int n;
  double h, inv_h;
  unsigned mask;             // mask + 1 buckets
  int* ccount;               // particles per bucket
  int* cfill;                // scatter cursor per bucket
  const long long* cstart;   // bucket starts (mask + 2 entries)
  GridEntry* entry;          // particles by bucket
  unsigned* cellh;           // bucket of each particle (large: unused)
  int* large;                // indices of large particles (any order)
  int* nlarge;
  // partners of a large particle are searched in chunks of `chunk`
  // candidates j (nchunks per particle, chunk c covers [c*chunk, (c+1)*chunk)),
  // one workgroup per (large particle, chunk); lcount[slot * nchunks + c] holds
  // each chunk's partner count
  int chunk, nchunks;
  int* lcount;
  // the first kBpKeep partners of each particle as the count pass found
  // them (discovery order), so that the fill pass only sorts them
  int* keep;
};

__device__ __forceinline__ bool is_large(const GridArgs& g, int i, const Aabb& b) {
  if (g.obstacle && g.obstacle[i]) return true;
  for (int q = 0; q < 3; ++q)
    if (!(b.hi[q] - b.lo[q] <= g.h)) return true;
  return false;
}

__global__ __launch_bounds__(256) void k_grid_bin(GridArgs g) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= g.n) return;
  const Aabb b = g.box[i];
  if (is_large(g, i, b)) {
    g.large[atomicAdd(g.nlarge, 1)] = i;
    return;
  }
  long long c[3];
  cell_of(b, g.inv_h, c);
  const unsigned hsh = hash_cell(c[0], c[1], c[2], g.mask);
  g.cellh[i] = hsh;
  atomicAdd(&g.ccount[hsh], 1);
}

__global__ __launch_bounds__(256) void k_grid_scatter(GridArgs g) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= g.n) return;
  GridEntry e;
  e.box = g.box[i];
  if (is_large(g, i, e.box)) return;
  const unsigned hsh = g.cellh[i];
  long long c[3];
  cell_of(e.box, g.inv_h, c);
  for (int q = 0; q < 3; ++q) e.cell[q] = static_cast<int>(c[q]);
  e.id = i;
  g.entry[g.cstart[hsh] + atomicAdd(&g.cfill[hsh], 1)] = e;
}

constexpr int kBpWaves = 4;    // particles per workgroup
constexpr int kBpList = 512;   // partners sorted in LDS per particle (else a serial sort)
constexpr int kBpKeep = 64;    // partners kept by the count pass per particle (one per lane)

// The partners j > i of a particle i that is not large, by L = 32 or 64 lanes
// of a wave (`active`: they have one): calls put(position, j) on the finding
// lane for every partner, positions 0.. in discovery order; returns their
// number.  27 lanes look up the neighbour cells' buckets; the buckets' members
// then form one list that all L lanes go through.  A member counts for the
// lane whose cell is its own, so that two cells that share a bucket do not find
// it twice.  The large particles are strided over the lanes.  Finds are
// compacted with ballots, so every lane sees the running count.
template <int L, typename F>
__device__ __forceinline__ int grid_partners(const GridArgs& g, int i, const Aabb& bi, bool active,
                                             int lane, F put) {
  const int sl = lane & (L - 1), first = lane - sl;
  auto part = [&](unsigned long long m) { return L == 64 ? m : (m >> first) & 0xffffffffull; };
  const unsigned long long below = (1ull << sl) - 1;
  long long c[3];
  cell_of(bi, g.inv_h, c);
  const bool walk = active && sl < 27;
  c[0] += sl / 9 - 1;
  c[1] += (sl / 3) % 3 - 1;
  c[2] += sl % 3 - 1;
  const unsigned hsh = hash_cell(c[0], c[1], c[2], g.mask);
  const int s0 = walk ? static_cast<int>(g.cstart[hsh]) : 0;
  const int len = walk ? static_cast<int>(g.cstart[hsh + 1]) - s0 : 0;
  int incl = len;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const int t = __shfl_up(incl, o, 32);
    if (sl >= o) incl += t;
  }
  const int excl = incl - len;  // lanes 27.. hold the total
  const int total = __shfl(incl, first + 31);
  int found = 0;
  for (int f0 = 0; __ballot(f0 < total); f0 += L) {
    const int f = f0 + sl;
    // the bucket of member f: the last of the 27 that starts at or before it
    int b = 0;
#pragma unroll
    for (int h = 16; h > 0; h >>= 1) {
      const int at = __shfl(excl, first + b + h);
      if (b + h < 27 && at <= f) b += h;
    }
    const int bs = __shfl(s0, first + b), be = __shfl(excl, first + b);
    const int cx = __shfl(static_cast<int>(c[0]), first + b);
    const int cy = __shfl(static_cast<int>(c[1]), first + b);
    const int cz = __shfl(static_cast<int>(c[2]), first + b);
    bool e = false;
    int cand = -1;
    if (f < total) {
      const GridEntry m = g.entry[bs + (f - be)];
      cand = m.id;
      e = cand > i && m.cell[0] == cx && m.cell[1] == cy && m.cell[2] == cz && overlap(bi, m.box);
    }
    const unsigned long long mask = part(__ballot(e));
    if (e) put(found + __popcll(mask & below), cand);
    found += __popcll(mask);
  }
  const int nl = *g.nlarge;
  for (int o0 = 0; o0 < nl; o0 += L) {
    const int o = o0 + sl;
    bool e = false;
    int cand = -1;
    if (active && o < nl) {
      cand = g.large[o];
      e = cand > i && overlap(bi, g.box[cand]);
    }
    const unsigned long long mask = part(__ballot(e));
    if (e) put(found + __popcll(mask & below), cand);
    found += __popcll(mask);
  }
  return found;
}

// Partners j of a large particle i in chunk c: every j > i of the chunk (not
// both obstacles), ascending, 1,024 a round over the workgroup's four waves;
// put(position, j) on the finding lane.  Returns their number.
template <typename F>
__device__ __forceinline__ int large_chunk(const GridArgs& g, int i, int c, int* wave_count,
                                           F put) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const Aabb bi = g.box[i];
  const bool obst_i = g.obstacle && g.obstacle[i];
  const int lo = c * g.chunk > i + 1 ? c * g.chunk : i + 1;
  const int hi = (c + 1) * g.chunk < g.n ? (c + 1) * g.chunk : g.n;
  int found = 0;
  for (int j0 = lo; j0 < hi; j0 += 256 * kBpWaves) {
    // four strips of 64 per wave: their loads are issued together
    bool e[4];
    int m = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = j0 + 256 * w + 64 * q + lane;
      e[q] = j < hi && !(obst_i && g.obstacle && g.obstacle[j]) && overlap(bi, g.box[j]);
      m += __popcll(__ballot(e[q]));
    }
    if (lane == 0) wave_count[w] = m;
    __syncthreads();
    int at = found;
    for (int o = 0; o < kBpWaves; ++o) {
      at += o < w ? wave_count[o] : 0;
      found += wave_count[o];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned long long mask = __ballot(e[q]);
      if (e[q]) put(at + lane_prefix(mask), j0 + 256 * w + 64 * q + lane);
      at += __popcll(mask);
    }
    __syncthreads();  // the next round overwrites the counts
  }
  return found;
}

// Large particles, one workgroup per (slot, chunk) item, strided over a
// persistent grid (the number of large particles is known on the device
// only): chunk partner counts.  Few items: the latency of a chunk's loads is
// what they cost (a wave per item, four rounds: 16 us in a hopper of 15,651
// particles, 7 us now; the fill 14 and 6).
__global__ __launch_bounds__(64 * kBpWaves) void k_large_count(GridArgs g) {
  __shared__ int wave_count[kBpWaves];
  const long long items = static_cast<long long>(*g.nlarge) * g.nchunks;
  for (long long t = blockIdx.x; t < items; t += gridDim.x) {
    const int o = static_cast<int>(t / g.nchunks), c = static_cast<int>(t - o * static_cast<long long>(g.nchunks));
    const int m = large_chunk(g, g.large[o], c, wave_count, [](int, int) {});
    if (threadIdx.x == 0) g.lcount[t] = m;
  }
}

// Partner count of each large particle: the sum of its chunk counts.
__global__ __launch_bounds__(64 * kBpWaves) void k_large_sum(GridArgs g, int* __restrict__ count) {
  const int lane = threadIdx.x & 63;
  const int nw = gridDim.x * kBpWaves;
  const int nl = *g.nlarge;
  for (int o = blockIdx.x * kBpWaves + (threadIdx.x >> 6); o < nl; o += nw) {
    int m = 0;
    for (int c = lane; c < g.nchunks; c += 64) m += g.lcount[static_cast<long long>(o) * g.nchunks + c];
    for (int k = 32; k > 0; k >>= 1) m += __shfl_xor(m, k);
    if (lane == 0) count[g.large[o]] = m;
  }
}

// Writes each chunk's partners after those of the particle's earlier chunks.
__global__ __launch_bounds__(64 * kBpWaves) void k_large_fill(GridArgs g,
                                                               const long long* __restrict__ start,
                                                               long long cap,
                                                               int* __restrict__ pairs) {
  __shared__ int wave_count[kBpWaves];
  const int lane = threadIdx.x & 63;
  const long long items = static_cast<long long>(*g.nlarge) * g.nchunks;
  for (long long t = blockIdx.x; t < items; t += gridDim.x) {
    const int o = static_cast<int>(t / g.nchunks), c = static_cast<int>(t - o * static_cast<long long>(g.nchunks));
    const int i = g.large[o];
    long long before = 0;
    for (int q = lane; q < c; q += 64) before += g.lcount[t - c + q];
    for (int k = 32; k > 0; k >>= 1) before += __shfl_xor(before, k);
    const long long s = start[i] + before;
    large_chunk(g, i, c, wave_count, [&](int pos, int j) {
      const long long q = s + pos;
      if (q < cap) {
        pairs[2 * q] = i;
        pairs[2 * q + 1] = j;
      }
    });
  }
}

// Partner counts, two particles per wave (the walk is latency bound: two
// searches share each round of dependent loads).
__global__ __launch_bounds__(64 * kBpWaves) void k_grid_count2(GridArgs g,
                                                                int* __restrict__ count) {
  const int lane = threadIdx.x & 63;
  const int i = (blockIdx.x * kBpWaves + (threadIdx.x >> 6)) * 2 + (lane >> 5);
  const bool valid = i < g.n;
  const Aabb bi = g.box[valid ? i : 0];
  const bool active = valid && !is_large(g, i, bi);
  int* kept = g.keep + static_cast<long long>(valid ? i : 0) * kBpKeep;
  auto keep = [&](int pos, int j) {
    if (pos < kBpKeep) kept[pos] = j;
  };
  const int m = grid_partners<32>(g, i, bi, active, lane, keep);
  // large particles: k_large_count / k_large_sum, launched after this
  if (valid && (lane & 31) == 0) count[i] = active ? m : 0;
}

// Writes the partners of i at start[i].. in ascending order (pairs beyond
// cap are not written).
__global__ __launch_bounds__(64 * kBpWaves) void k_grid_fill(GridArgs g,
                                                              const long long* __restrict__ start,
                                                              long long cap,
                                                              int* __restrict__ pairs) {
  __shared__ int list[kBpWaves][kBpList];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * kBpWaves + w;
  if (i >= g.n) return;  // wave-uniform
  const long long s = start[i];
  const long long m = start[i + 1] - s;
  const Aabb bi = g.box[i];
  auto direct = [&](int pos, int j) {
    const long long q = s + pos;
    if (q < cap) {
      pairs[2 * q] = i;
      pairs[2 * q + 1] = j;
    }
  };
  if (is_large(g, i, bi)) return;  // k_large_fill
  if (m <= kBpKeep) {
    // the count pass kept them all: lane e ranks entry e among the m
    // (distinct) partners by shuffles and writes it in place
    const int v = lane < m ? g.keep[static_cast<long long>(i) * kBpKeep + lane] : 0;
    int rank = 0;
    for (int q = 0; q < m; ++q) {
      const int u = __shfl(v, q);
      rank += u < v ? 1 : 0;
    }
    if (lane < m) direct(rank, v);
    return;
  }
  if (m > kBpList) {
    // more partners than the LDS list holds: unsorted, then a serial sort
    grid_partners<64>(g, i, bi, true, lane, direct);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
    if (lane == 0) {
      const long long e = s + m < cap ? s + m : cap;
      for (long long a = s + 1; a < e; ++a) {
        const int v = pairs[2 * a + 1];
        long long b = a - 1;
        while (b >= s && pairs[2 * b + 1] > v) {
          pairs[2 * (b + 1) + 1] = pairs[2 * b + 1];
          --b;
        }
        pairs[2 * (b + 1) + 1] = v;
      }
    }
    return;
  }
  int* lst = list[w];
  const int found = grid_partners<64>(g, i, bi, true, lane, [&](int pos, int j) {
    if (pos < kBpList) lst[pos] = j;
  });
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
  const int mm = found < kBpList ? found : kBpList;
  // partners are distinct: the rank of v is the number of smaller partners
  for (int e = lane; e < mm; e += 64) {
    const int v = lst[e];
    int rank = 0;
    for (int q = 0; q < mm; ++q) rank += lst[q] < v ? 1 : 0;
    direct(rank, v);
  }
}

// Scenes of at most kSmallScene particles: every pair (i < j) tested, in place
// of the grid's dozen launches.  Up to kOneGroupScene of them by this one
// workgroup of 16 waves (65 particles: 8 us; 1,001 particles took it 400 us).  The same
// candidate set (boxes overlap, not both obstacles) in the same order (i
// ascending, then j ascending), with the same outputs: start[0..n] (start[n]
// the total, which may exceed cap) and the pairs that fit cap.  A wave per
// particle i sweeps j > i in strips of 64: counts, their prefix sums, then
// the same sweep writes each partner at start[i] + its rank.
constexpr int kSmallScene = 1024;
constexpr int kOneGroupScene = 128;

__global__ __launch_bounds__(1024) void k_small_pairs(const Aabb* __restrict__ box,
                                                      const int* __restrict__ obstacle, int n,
                                                      long long* __restrict__ start,
                                                      long long cap, int* __restrict__ pairs) {
  // the boxes and obstacle flags staged once: both sweeps read LDS only
  __shared__ Aabb s_box[kOneGroupScene];
  __shared__ unsigned char s_obst[kOneGroupScene];
  __shared__ long long s_start[kOneGroupScene + 1];
  __shared__ long long s_wave[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = threadIdx.x;
  if (t < n) {
    s_box[t] = box[t];
    s_obst[t] = obstacle && obstacle[t] ? 1 : 0;
  }
  __syncthreads();
  for (int i = w; i < n; i += 16) {
    const Aabb bi = s_box[i];
    const bool oi = s_obst[i] != 0;
    int m = 0;
    for (int j0 = i + 1; j0 < n; j0 += 64) {
      const int j = j0 + lane;
      const bool e = j < n && !(oi && s_obst[j]) && overlap(bi, s_box[j]);
      m += __popcll(__ballot(e));
    }
    if (lane == 0) s_start[i] = m;
  }
  __syncthreads();
  // exclusive prefix sums: one count per thread, waves, then wave totals
  const long long c = t < n ? s_start[t] : 0;
  long long incl = c;
  for (int o = 1; o < 64; o <<= 1) {
    const long long u = __shfl_up(incl, o);
    incl += lane >= o ? u : 0;
  }
  if (lane == 63) s_wave[w] = incl;
  __syncthreads();
  long long before = 0;
  for (int q = 0; q < w; ++q) before += s_wave[q];
  const long long excl = before + incl - c;
  if (t < n) {
    s_start[t] = excl;
    start[t] = excl;
  }
  if (t == (n > 0 ? n - 1 : 0)) {
    s_start[n] = n > 0 ? excl + c : 0;
    start[n] = n > 0 ? excl + c : 0;
  }
  __syncthreads();
  for (int i = w; i < n; i += 16) {
    const Aabb bi = s_box[i];
    const bool oi = s_obst[i] != 0;
    const long long s0 = s_start[i];
    int found = 0;
    for (int j0 = i + 1; j0 < n; j0 += 64) {
      const int j = j0 + lane;
      const bool e = j < n && !(oi && s_obst[j]) && overlap(bi, s_box[j]);
      const unsigned long long mask = __ballot(e);
      const long long q = s0 + found + lane_prefix(mask);
      if (e && q < cap) {
        pairs[2 * q] = i;
        pairs[2 * q + 1] = j;
      }
      found += __popcll(mask);
    }
  }
}

// The same set for more particles (to kSmallScene): a wave per particle i
// sweeps j > i, once for the counts and, after their scan, once more for the
// pairs: start[0..n] and the pairs that fit cap.  1,001 particles: 11 + 5 +
// 11 us, 129: 14 us in all (15.5 us by the one workgroup, 8 us at 65: the line
// lies where the two more launches are paid back).
template <bool kFill>
__global__ __launch_bounds__(256) void k_all_pairs(const Aabb* __restrict__ box,
                                                   const int* __restrict__ obstacle, int n,
                                                   int* __restrict__ count,
                                                   const long long* __restrict__ start,
                                                   long long cap, int* __restrict__ pairs) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + static_cast<int>(threadIdx.x >> 6);
  if (i >= n) return;  // wave-uniform
  const Aabb bi = box[i];
  const bool oi = obstacle && obstacle[i];
  const long long s0 = kFill ? start[i] : 0;
  int found = 0;
  for (int j0 = i + 1; j0 < n; j0 += 64) {
    const int j = j0 + lane;
    const bool e = j < n && !(oi && obstacle[j]) && overlap(bi, box[j]);
    const unsigned long long mask = __ballot(e);
    const long long q = s0 + found + lane_prefix(mask);
    if (kFill && e && q < cap) {
      pairs[2 * q] = i;
      pairs[2 * q + 1] = j;
    }
    found += __popcll(mask);
  }
  if (!kFill && lane == 0) count[i] = found;
}

int scan_counts(const int* counts, int n, long long* offs, hipStream_t st);
int scan_counts_with(const int* counts, int n, long long* offs, long long* sums,
                     hipStream_t st);
int scan_sums_len(int n);
int scan_reserve(int n);

struct BpScratch {
  DevBuf box, ccount, cfill, cstart, entry, cellh, count, start, err, obst, lcount, keep, cbox,
      sph;
};
static BpScratch g_bp;

// Candidates per large-particle chunk: 1024 (one round of a workgroup), more
// for very large n so that a particle has at most 256 chunks.
static int large_chunk_len(int n) {
  int c = 1024;
  while (static_cast<long long>(c) * 256 < n) c *= 2;
  return c;
}

static int large_chunks(int n) {
  const int c = large_chunk_len(n);
  return (n + c - 1) / c > 0 ? (n + c - 1) / c : 1;
}

// Persistent grid of the large-particle kernels.
static unsigned large_grid(long long items) {
  return static_cast<unsigned>(items < 1 ? 1 : (items > 2048 ? 2048 : items));
}

static unsigned table_size(int n) {
  unsigned tbl = 1;
  while (tbl < 2u * static_cast<unsigned>(n)) tbl <<= 1;
  return tbl;
}

// The device buffers of one broad phase over n particles and ntri
// triangles (entries of each, in order of the layout below).
struct BpBuffers {
  Aabb* box;           // n + 1
  Aabb* cbox;          // ntri / 64 + n + 1
  int* ccount;         // tbl + 1
  int* cfill;          // tbl
  long long* cstart;   // tbl + 1
  GridEntry* entry;    // n + 1
  unsigned* cellh;     // n + 1
  int* count;          // n + 1
  long long* start;    // n + 1
  int* nlarge;         // 1
  int* large;          // n + 1
  int* lcount;         // (n + 1) * large_chunks(n)
  int* keep;           // (n + 1) * kBpKeep
  long long* sums;     // scan_sums_len(max(tbl, n)); null: the scan's own scratch
  double* sph;         // 4 (n + 1): bounding spheres (centre, radius); may be null
};

static BpBuffers library_buffers() {
  return BpBuffers{g_bp.box.as<Aabb>(),     g_bp.cbox.as<Aabb>(),    g_bp.ccount.as<int>(),
                   g_bp.cfill.as<int>(),    g_bp.cstart.as<long long>(), g_bp.entry.as<GridEntry>(),
                   g_bp.cellh.as<unsigned>(), g_bp.count.as<int>(),  g_bp.start.as<long long>(),
                   g_bp.err.as<int>(),      g_bp.obst.as<int>(),     g_bp.lcount.as<int>(),
                   g_bp.keep.as<int>(),     nullptr,                 g_bp.sph.as<double>()};
}

static int scan_into(const BpBuffers& b, const int* counts, int n, long long* offs,
                     hipStream_t st) {
  return b.sums ? scan_counts_with(counts, n, offs, b.sums, st) : scan_counts(counts, n, offs, st);
}

// The particle boxes of the last broad phase (lo xyz, hi xyz per particle:
// the vertex box inflated by the margin and 0.5e-9 m), valid until the next
// call on more particles.
const double* broadphase_boxes() { return g_bp.box.as<double>(); }
const double* broadphase_block_boxes() { return g_bp.cbox.as<double>(); }
// The particles' bounding spheres (x, y, z, r) of the last broad phase.
const double* broadphase_spheres() { return g_bp.sph.as<double>(); }

// The same boxes for the current geometry, without the grid (for callers
// of the detection that did not run the broad phase).
int particle_boxes(const dh_geometry* geom, const double** out, hipStream_t st) {
  const int n = geom->nparticles;
  int rc;
  if ((rc = g_bp.box.grow(sizeof(Aabb) * (n + 1)))) return rc;
  if ((rc = g_bp.cbox.grow(sizeof(Aabb) * ((geom->ntri_total + 63) / 64 + n + 1)))) return rc;
  if ((rc = g_bp.sph.grow(sizeof(double) * 4 * (n + 1)))) return rc;
  if (n > 0)
    launch_aabb(geom, g_bp.box.as<Aabb>(), g_bp.cbox.as<Aabb>(), g_bp.sph.as<double>(), st);
  DH_HIP_CHECK(hipGetLastError());
  *out = g_bp.box.as<double>();
  return DH_OK;
}

// Buffers of the broad phase for n particles (call before a capture).
int broadphase_reserve(int n, int ntri) {
  int rc;
  const unsigned tbl = table_size(n);
  if ((rc = g_bp.box.grow(sizeof(Aabb) * (n + 1)))) return rc;
  if ((rc = g_bp.cbox.grow(sizeof(Aabb) * ((ntri + 63) / 64 + n + 1)))) return rc;
  if ((rc = g_bp.sph.grow(sizeof(double) * 4 * (n + 1)))) return rc;
  if ((rc = g_bp.ccount.grow(sizeof(int) * (tbl + 1)))) return rc;
  if ((rc = g_bp.cfill.grow(sizeof(int) * tbl))) return rc;
  if ((rc = g_bp.cstart.grow(sizeof(long long) * (tbl + 1)))) return rc;
  if ((rc = g_bp.entry.grow(sizeof(GridEntry) * (n + 1)))) return rc;
  if ((rc = g_bp.cellh.grow(sizeof(unsigned) * (n + 1)))) return rc;
  if ((rc = g_bp.count.grow(sizeof(int) * (n + 1)))) return rc;
  if ((rc = g_bp.start.grow(sizeof(long long) * (n + 1)))) return rc;
  if ((rc = g_bp.err.grow(sizeof(int)))) return rc;
  if ((rc = g_bp.obst.grow(sizeof(int) * (n + 1)))) return rc;
  // every particle may be large (a cell smaller than the particles)
  if ((rc = g_bp.lcount.grow(sizeof(int) * static_cast<size_t>(n + 1) * large_chunks(n))))
    return rc;
  if ((rc = g_bp.keep.grow(sizeof(int) * static_cast<size_t>(n + 1) * kBpKeep))) return rc;
  return scan_reserve(static_cast<int>(tbl) > n ? static_cast<int>(tbl) : n);
}

// Clears the counters the grid passes add to (fill kernels, no memset, so
// that captured work may contain it).
static void grid_clear(const BpBuffers& b, unsigned tbl, hipStream_t st) {
  zero_async(ZeroRegions{{reinterpret_cast<unsigned*>(b.nlarge),
                          reinterpret_cast<unsigned*>(b.ccount),
                          reinterpret_cast<unsigned*>(b.cfill), nullptr},
                         {1, static_cast<long long>(tbl), static_cast<long long>(tbl), 0}},
             st);
}

// Boxes, the sorted cell list and the partner counts, on cleared counters.
static int grid_build(const dh_geometry* geom, const int* obstacle_dev, double cell,
                      const BpBuffers& b, GridArgs& g, hipStream_t st) {
  const int n = geom->nparticles;
  const unsigned tbl = table_size(n);
  launch_aabb(geom, b.box, b.cbox, b.sph, st);
  g.box = b.box;
  g.obstacle = obstacle_dev;
  g.n = n;
  g.h = cell;
  g.inv_h = 1.0 / cell;
  g.mask = tbl - 1;
  g.ccount = b.ccount;
  g.cfill = b.cfill;
  g.cstart = b.cstart;
  g.entry = b.entry;
  g.cellh = b.cellh;
  g.large = b.large;
  g.nlarge = b.nlarge;
  g.chunk = large_chunk_len(n);
  g.nchunks = large_chunks(n);
  g.lcount = b.lcount;
  g.keep = b.keep;
  hipLaunchKernelGGL(k_grid_bin, grid_for(n, 256), 256, 0, st, g);
  int rc;
  if ((rc = scan_into(b, b.ccount, static_cast<int>(tbl), b.cstart, st))) return rc;
  hipLaunchKernelGGL(k_grid_scatter, grid_for(n, 256), 256, 0, st, g);
  hipLaunchKernelGGL(k_grid_count2, grid_for(n, 2 * kBpWaves), 64 * kBpWaves, 0, st, g, b.count);
  const long long items = static_cast<long long>(n) * g.nchunks;  // bound on the device count
  hipLaunchKernelGGL(k_large_count, large_grid(items), 64 * kBpWaves, 0, st, g);
  hipLaunchKernelGGL(k_large_sum, large_grid((n + kBpWaves - 1) / kBpWaves), 64 * kBpWaves, 0, st, g, b.count);
  DH_HIP_CHECK(hipGetLastError());
  return scan_into(b, b.count, n, b.start, st);
}

static void grid_fill(const GridArgs& g, const BpBuffers& b, long long cap, int* pairs,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_grid_fill, grid_for(g.n, kBpWaves), 64 * kBpWaves, 0, st, g, b.start, cap,
                     pairs);
  hipLaunchKernelGGL(k_large_fill, large_grid(static_cast<long long>(g.n) * g.nchunks),
                     64 * kBpWaves, 0, st, g, b.start, cap, pairs);
}

// The broad phase of at most kSmallScene particles: nothing is written past
// cap, so the pairs come with the count.
static int small_pairs(const dh_geometry* geom, const int* obstacle_dev, const BpBuffers& b,
                       int* pairs, long long cap, hipStream_t st) {
  const int n = geom->nparticles;
  if (n > 0) launch_aabb(geom, b.box, b.cbox, b.sph, st);
  if (n <= kOneGroupScene) {
    hipLaunchKernelGGL(k_small_pairs, 1, 1024, 0, st, b.box, obstacle_dev, n, b.start, cap, pairs);
  } else {
    const unsigned grid = grid_for(n, 4);
    hipLaunchKernelGGL(k_all_pairs<false>, grid, 256, 0, st, b.box, obstacle_dev, n, b.count,
                       b.start, cap, pairs);
    int rc;
    if ((rc = scan_into(b, b.count, n, b.start, st))) return rc;
    hipLaunchKernelGGL(k_all_pairs<true>, grid, 256, 0, st, b.box, obstacle_dev, n, b.count,
                       b.start, cap, pairs);
  }
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

// The eager broad phase on the buffers b: the total is read back (through the
// library's pinned mailbox, or by a copy where nothing may be allocated), and
// the pairs are written only if it fits cap.
static int broadphase_run(const dh_geometry* geom, const int* obstacle_dev, double cell,
                          const BpBuffers& b, bool mailbox, int* pairs, long long cap,
                          long long* npairs, hipStream_t st) {
  auto read_total = [&](long long* total) -> int {
    if (mailbox) return read_back(b.start + geom->nparticles, 2, total, st);
    DH_HIP_CHECK(hipMemcpyAsync(total, b.start + geom->nparticles, sizeof(long long),
                                hipMemcpyDeviceToHost, st));
    DH_HIP_CHECK(hipStreamSynchronize(st));
    return DH_OK;
  };
  const int n = geom->nparticles;
  if (n <= kSmallScene) {
    int rc;
    if (n > 0 && (rc = small_pairs(geom, obstacle_dev, b, pairs, cap, st))) return rc;
    long long total = 0;
    if (n > 0 && (rc = read_total(&total))) return rc;
    *npairs = total;
    return total > cap ? DH_ERR_CAPACITY : DH_OK;
  }
  grid_clear(b, table_size(n), st);
  GridArgs g;
  int rc;
  if ((rc = grid_build(geom, obstacle_dev, cell, b, g, st))) return rc;
  long long total = 0;
  if ((rc = read_total(&total))) return rc;
  *npairs = total;
  if (*npairs > cap) return DH_ERR_CAPACITY;
  grid_fill(g, b, cap, pairs, st);
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

int broadphase_impl(const dh_geometry* geom, const int* obstacle_dev, double cell, int* pairs,
                    long long cap, long long* npairs, hipStream_t st) {
  int rc;
  if ((rc = broadphase_reserve(geom->nparticles, geom->ntri_total))) return rc;
  return broadphase_run(geom, obstacle_dev, cell, library_buffers(), true, pairs, cap, npairs, st);
}

// The broad phase for a captured step: the same kernels with no host
// read-back.  *np_dev (the total, which may exceed cap) is left at the
// returned device address; pairs beyond cap are not written.
int broadphase_graph(const dh_geometry* geom, const int* obstacle_dev, double cell, int* pairs,
                     long long cap, const long long** np_dev, hipStream_t st) {
  const int n = geom->nparticles;
  int rc;
  if ((rc = broadphase_reserve(n, geom->ntri_total))) return rc;
  const BpBuffers b = library_buffers();
  *np_dev = b.start + n;
  if (n <= kSmallScene) return small_pairs(geom, obstacle_dev, b, pairs, cap, st);
  grid_clear(b, table_size(n), st);
  GridArgs g;
  if ((rc = grid_build(geom, obstacle_dev, cell, b, g, st))) return rc;
  grid_fill(g, b, cap, pairs, st);
  DH_HIP_CHECK(hipGetLastError());
  return DH_OK;
}

// ------------------------------------------------ broad phase, no allocation
// One statically allocated device array holds every buffer of a broad phase
// of at most DH_NOALLOC_BP_PARTICLES particles and DH_NOALLOC_BP_TRIANGLES
// triangles (8,523,264 bytes).  Each device keeps its own copy for the life of
// the process; every call on a device shares it, so calls that overlap on one
// device race.
constexpr size_t kNaAlign = 256;

static size_t na_round(size_t b) { return (b + kNaAlign - 1) / kNaAlign * kNaAlign; }

// Carves the buffers of (n, ntri) out of base; returns the bytes used.
static size_t noalloc_layout(char* base, int n, int ntri, BpBuffers* b) {
  const size_t tbl = table_size(n);
  const size_t np1 = static_cast<size_t>(n) + 1;
  const int scan_n = static_cast<int>(tbl) > n ? static_cast<int>(tbl) : n;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* p = base ? base + off : nullptr;
    off += na_round(bytes);
    return p;
  };
  BpBuffers t;
  t.box = reinterpret_cast<Aabb*>(take(sizeof(Aabb) * np1));
  // the chunk boxes, which only the detection reads, are not kept here: their
  // place holds the grid's entries
  t.cbox = nullptr;
  const size_t chunks = sizeof(Aabb) * ((ntri + 63) / 64 + np1), entries = sizeof(GridEntry) * np1;
  t.entry = reinterpret_cast<GridEntry*>(take(chunks > entries ? chunks : entries));
  t.ccount = reinterpret_cast<int*>(take(sizeof(int) * (tbl + 1)));
  t.cfill = reinterpret_cast<int*>(take(sizeof(int) * tbl));
  t.cstart = reinterpret_cast<long long*>(take(sizeof(long long) * (tbl + 1)));
  take(sizeof(int) * np1);  // unused: the array's published size is kept
  t.cellh = reinterpret_cast<unsigned*>(take(sizeof(unsigned) * np1));
  t.count = reinterpret_cast<int*>(take(sizeof(int) * np1));
  t.start = reinterpret_cast<long long*>(take(sizeof(long long) * np1));
  t.nlarge = reinterpret_cast<int*>(take(sizeof(int)));
  t.large = reinterpret_cast<int*>(take(sizeof(int) * np1));
  t.lcount = reinterpret_cast<int*>(take(sizeof(int) * np1 * large_chunks(n)));
  t.keep = reinterpret_cast<int*>(take(sizeof(int) * np1 * kBpKeep));
  t.sums = reinterpret_cast<long long*>(take(sizeof(long long) * scan_sums_len(scan_n)));
  t.sph = nullptr;  // the detection's sphere test is not part of this entry point
  if (b) *b = t;
  return off;
}

// Bytes of the largest layout (every buffer grows with n and ntri).
constexpr size_t kNaScratchBytes = 8523264;

__device__ __align__(256) char scratch[kNaScratchBytes];

constexpr int kMaxDevices = 64;
static void* g_na_ptr[kMaxDevices];
static std::mutex g_na_mu;

// The device address of this device's `scratch` (looked up on the first
// call on each device, with that device current).
static int noalloc_scratch(char** out) {
  int dev = 0;
  DH_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices)
    return set_error(DH_ERR_UNSUPPORTED, "dh_broadphase_noalloc: device %d", dev);
  std::lock_guard<std::mutex> lock(g_na_mu);
  if (!g_na_ptr[dev]) {
    void* p = nullptr;
    DH_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_na_ptr[dev] = p;
  }
  *out = static_cast<char*>(g_na_ptr[dev]);
  return DH_OK;
}

}  // namespace dh

using namespace dh;

extern "C" int dh_broadphase(const dh_geometry* geom, const int* obstacle_dev, double cell,
                             int* pairs_dev, int cap, int* npairs, void* stream) {
  int rc = ensure_init();
  if (rc) return rc;
  if (!geom || !npairs || !(cell > 0) || cap < 0 || (cap > 0 && !pairs_dev))
    return set_error(DH_ERR_ARG, "dh_broadphase: bad arguments");
  *npairs = 0;
  if (geom->nparticles < 2) return DH_OK;
  long long np = 0;
  rc = broadphase_impl(geom, obstacle_dev, cell, pairs_dev, cap, &np, as_stream(stream));
  *npairs = static_cast<int>(np);
  return rc;
}

extern "C" int dh_broadphase_noalloc(const dh_geometry* geom, const int* obstacle_dev,
                                     double cell, int* pairs_dev, int cap, int* npairs,
                                     void* stream) {
  int rc = ensure_init();
  if (rc) return rc;
  if (!geom || !npairs || !(cell > 0) || cap < 0 || (cap > 0 && !pairs_dev) ||
      geom->nparticles < 0 || geom->ntri_total < 0)
    return set_error(DH_ERR_ARG, "dh_broadphase_noalloc: bad arguments");
  *npairs = 0;
  if (geom->nparticles > DH_NOALLOC_BP_PARTICLES || geom->ntri_total > DH_NOALLOC_BP_TRIANGLES)
    return set_error(DH_ERR_CAPACITY,
                     "dh_broadphase_noalloc: %d particles / %d triangles exceed the fixed "
                     "scratch (at most %d / %d)",
                     geom->nparticles, geom->ntri_total, DH_NOALLOC_BP_PARTICLES,
                     DH_NOALLOC_BP_TRIANGLES);
  if (geom->nparticles < 2) return DH_OK;
  char* base = nullptr;
  if ((rc = noalloc_scratch(&base))) return rc;
  BpBuffers b;
  if (noalloc_layout(base, geom->nparticles, geom->ntri_total, &b) > kNaScratchBytes)
    return set_error(DH_ERR_CAPACITY, "dh_broadphase_noalloc: scratch layout too large");
  long long np = 0;
  rc = broadphase_run(geom, obstacle_dev, cell, b, false, pairs_dev, cap, &np, as_stream(stream));
  *npairs = static_cast<int>(np);
  return rc;
}

// Bytes the fixed scratch must hold for the largest accepted sizes (a
// build-time check of kNaScratchBytes, exported for tests).
extern "C" size_t dh_broadphase_noalloc_scratch_bytes(int nparticles, int ntri) {
  return noalloc_layout(nullptr, nparticles, ntri, nullptr);
}
