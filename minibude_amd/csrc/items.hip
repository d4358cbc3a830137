// items.hip -- exact pose energies from sorted items.
//
// An item is one ligand atom under one pose.  Its energy is a sum over the
// protein atoms of three hinges that are exactly zero beyond a few Angstrom
// (pair_reach), about 2 % of the pairs in a protein of 4,096 atoms.  A
// wave can leave a protein atom out only when it is out of reach of all its
// items, and 64 poses of one ligand atom lie all over the protein; so the
// items are first sorted by (forcefield type of the ligand atom, cell of
// space), and a wave then scores 64 x RB neighbouring items of one type
// against the protein atoms within reach of their box.  The pairs left out
// add fma(w, 0, e) == e; the others are summed in the same order by the
// same code as the tiled kernels' (fasten_core.h), and the energies of a
// pose's atoms are added in the ligand's order, so an energy is the tiled
// kernels' bit for bit however the items fell.
//
// One pass, per chunk of the plan:
//   prep_kernel    pose transforms, and the box of the translations
//   bin_kernel<0>  per (type, block of poses): items per cell, from LDS counts
//   column_kernel  those counts summed over the blocks, per (type, cell)
//   scan_kernel    the first item of every (type, cell)
//   bin_kernel<1>  items (x, y, z, where its energy goes) into their places
//   score_kernel   the items' energies
//   reduce_kernel  pose energies, the atoms' energies in order
// An item's place within its cell is whichever atomic came first; nothing an
// item's energy is made of depends on it.
//
// Measured against the tiled kernel on the same deck (device time): 4,096 x
// 64 atoms x 1,048,576 poses 79.4 -> 4.3 ms (items into place 0.8, counts
// 0.12, reduction 0.06, the rest the score kernel); 2,672 x 2,672 x 65,536
// 289 -> 9.1 ms; 938 x 26 x 65,536 1,030 -> 128 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>

#include "fasten_core.h"
#include "items.h"

namespace bude {
namespace items {

namespace {

using namespace core;

constexpr int kThreads = 1024;      // of the prep and bin kernels
constexpr int kCells = 4096;        // 16 per axis
constexpr int kMaxBounds = 256;     // work-groups of the prep kernel

struct Block {
  int64_t pose_off;      // row of the block's first pose
  uint32_t part_off;     // partial of (atom 0, first pose)
  uint32_t part_stride;  // from one atom to the next
  int32_t npose, natlig;
  uint32_t xf_off;       // first transform
  int32_t seg_pose;      // the first pose's place in its segment
};
static_assert(sizeof(Block) == 32, "Block is 32 bytes");

// The atoms of one type in one block: one row of the counts.
struct Row {
  int32_t block, atom0, natoms, slot;
};

// Rows ref[ref0 .. ref0 + nref) of one block, for one work-group.
struct Task {
  int32_t block, ref0, nref, pad;
};

struct Space {
  float lo[3], hi[3];  // where an item can have an energy
  float radius;        // of the ligand atoms about their frame's origin
};

__device__ __forceinline__ float wave_min(float v) {
  for (int d = 32; d; d >>= 1) v = fminf(v, __shfl_xor(v, d));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  for (int d = 32; d; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
  return v;
}

// Transforms of every pose of the chunk, and per work-group the box of its
// poses' translations (bounds[group]: three minima, three maxima).
__global__ __launch_bounds__(kThreads) void prep_kernel(const Block *__restrict__ blocks, int nblocks,
                                                        const float *__restrict__ poses, size_t stride,
                                                        const uint32_t *__restrict__ index, float4 *__restrict__ xf,
                                                        size_t nxf, float *__restrict__ bounds) {
  __shared__ float part[kThreads / 64][6];
  float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (int b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const Block bk = blocks[b];
    for (int j = threadIdx.x; j < bk.npose; j += kThreads) {
      const size_t row = size_t(bk.pose_off) + size_t(j);
      size_t q = row;
      if (index) q = size_t(bk.pose_off - bk.seg_pose) + index[row];
      const Xform t = make_xform(poses, stride, q);
      const size_t i = size_t(bk.xf_off) + size_t(j);
      xf[i] = make_float4(t.m[0], t.m[1], t.m[2], t.m[3]);
      xf[nxf + i] = make_float4(t.m[4], t.m[5], t.m[6], t.m[7]);
      xf[2 * nxf + i] = make_float4(t.m[8], t.m[9], t.m[10], t.m[11]);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        lo[k] = fminf(lo[k], t.m[4 * k + 3]);
        hi[k] = fmaxf(hi[k], t.m[4 * k + 3]);
      }
    }
  }
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float a = wave_min(lo[k]), b = wave_max(hi[k]);
    if ((threadIdx.x & 63) == 0) {
      part[wave][k] = a;
      part[wave][3 + k] = b;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    float v = part[0][threadIdx.x];
    for (int w = 1; w < kThreads / 64; w++)
      v = threadIdx.x < 3 ? fminf(v, part[w][threadIdx.x]) : fmaxf(v, part[w][threadIdx.x]);
    bounds[size_t(blockIdx.x) * 6 + threadIdx.x] = v;
  }
}

// 16 cells per axis over the box of the chunk's items (the translations'
// box widened by the ligands' radius) where it meets the scene's.
struct CellGrid {
  float lo[3], inv[3];
};

__device__ __forceinline__ CellGrid cell_grid(const float *__restrict__ bounds, int nbounds, const Space &sp,
                                              float *red /* LDS, 6 */) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // waves 0-2 the minima, 3-5 the maxima
  if (wave < 6) {
    float v = wave < 3 ? FLT_MAX : -FLT_MAX;
    for (int i = lane; i < nbounds; i += 64) {
      const float x = bounds[size_t(i) * 6 + wave];
      v = wave < 3 ? fminf(v, x) : fmaxf(v, x);
    }
    v = wave < 3 ? wave_min(v) : wave_max(v);
    if (lane == 0) red[wave] = v;
  }
  __syncthreads();
  CellGrid g;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float a = fmaxf(red[k] - sp.radius, sp.lo[k]), b = fminf(red[3 + k] + sp.radius, sp.hi[k]);
    g.lo[k] = a;
    g.inv[k] = b > a ? 16.0f / (b - a) : 0.0f;
  }
  return g;
}

// (clamped to the grid; NaN falls into cell 0 of its axis)
__device__ __forceinline__ uint32_t axis_cell(float x, float lo, float inv) {
  return uint32_t(__builtin_amdgcn_fmed3f((x - lo) * inv, 0.0f, 15.0f));
}

// Cells are numbered along a Hilbert curve: consecutive cells share a face,
// so items that straddle cells keep a small box (in Morton order a step can
// cross the whole grid; 9 % fewer atoms per item over 4,096 x 64 atoms x
// 1,048,576 poses, 16 % with a sixteenth of the poses).  Steps of Skilling's transform ("Programming the Hilbert
// curve", AIP Conf. Proc. 707, 2004) for a 16^3 grid.
constexpr uint16_t hilbert_place(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t v[3] = {x, y, z};
  for (uint32_t q = 8; q > 1; q >>= 1)
    for (int i = 0; i < 3; i++) {
      if (v[i] & q) {
        v[0] ^= q - 1;
      } else {
        const uint32_t t = (v[0] ^ v[i]) & (q - 1);
        v[0] ^= t;
        v[i] ^= t;
      }
    }
  v[1] ^= v[0];
  v[2] ^= v[1];
  uint32_t t = 0;
  for (uint32_t q = 8; q > 1; q >>= 1)
    if (v[2] & q) t ^= q - 1;
  uint32_t h = 0;
  for (int b = 3; b >= 0; b--)
    for (int i = 0; i < 3; i++) h = h << 1 | (((v[i] ^ t) >> b) & 1);
  return uint16_t(h);
}

struct Curve {
  uint16_t place[kCells];
};
constexpr Curve make_curve() {
  Curve c{};
  for (uint32_t i = 0; i < uint32_t(kCells); i++) c.place[i] = hilbert_place(i & 15, (i >> 4) & 15, i >> 8);
  return c;
}
__device__ const Curve kCurve = make_curve();

// curve: kCurve's places, in LDS.
__device__ __forceinline__ uint32_t cell_of(const CellGrid &g, const uint16_t *curve, float x, float y, float z) {
  return curve[axis_cell(x, g.lo[0], g.inv[0]) | axis_cell(y, g.lo[1], g.inv[1]) << 4 |
               axis_cell(z, g.lo[2], g.inv[2]) << 8];
}

// SCATTER 0: counts of each row's items per cell.  SCATTER 1: each item into
// its place.  One work-group per task, PPT poses per work-item.  Both read
// the same transforms and place items by the same explicit operations, so an
// item's cell is the same in both.
template <int PPT, int SCATTER>
__global__ __launch_bounds__(kThreads) void bin_kernel(const Task *__restrict__ tasks, const Block *__restrict__ blocks,
                                                       const int32_t *__restrict__ refs, const Row *__restrict__ rows,
                                                       const float4 *__restrict__ atoms,
                                                       const float4 *__restrict__ xf, size_t nxf,
                                                       const float *__restrict__ bounds, int nbounds, const Space sp,
                                                       int bits, uint32_t *__restrict__ hist,
                                                       const uint32_t *__restrict__ base, float4 *__restrict__ items) {
  __shared__ uint32_t h[kCells];
  __shared__ uint16_t curve[kCells];
  __shared__ float red[6];
  for (int i = threadIdx.x; i < kCells; i += kThreads) curve[i] = kCurve.place[i];  // (cell_grid waits for it)
  const CellGrid g = cell_grid(bounds, nbounds, sp, red);
  const Task t = tasks[blockIdx.x];
  const Block bk = blocks[t.block];
  const int ncells = 1 << bits, shift = 12 - bits;
  float4 m0[PPT], m1[PPT], m2[PPT];
#pragma unroll
  for (int k = 0; k < PPT; k++) {
    const int j = int(threadIdx.x) + k * kThreads;
    const size_t i = size_t(bk.xf_off) + size_t(j < bk.npose ? j : 0);
    m0[k] = xf[i];
    m1[k] = xf[nxf + i];
    m2[k] = xf[2 * nxf + i];
  }
  for (int r = 0; r < t.nref; r++) {
    const int id = refs[t.ref0 + r];
    const Row row = rows[id];
    uint32_t *hr = hist + size_t(id) * size_t(ncells);
    const uint32_t *br = base + size_t(row.slot) * size_t(ncells);
    for (int c = threadIdx.x; c < ncells; c += kThreads) h[c] = SCATTER ? br[c] + hr[c] : 0u;
    __syncthreads();
    for (int a = 0; a < row.natoms; a++) {
      const float4 la = atoms[row.atom0 + a];  // w bits: the atom's place in its ligand
      const uint32_t out = bk.part_off + uint32_t(__float_as_int(la.w)) * bk.part_stride;
#pragma unroll
      for (int k = 0; k < PPT; k++) {
        const int j = int(threadIdx.x) + k * kThreads;
        const float x = place(m0[k].x, m0[k].y, m0[k].z, m0[k].w, la);
        const float y = place(m1[k].x, m1[k].y, m1[k].z, m1[k].w, la);
        const float z = place(m2[k].x, m2[k].y, m2[k].z, m2[k].w, la);
        if (j < bk.npose) {
          const uint32_t c = cell_of(g, curve, x, y, z) >> shift;
          const uint32_t at = atomicAdd(&h[c], 1u);
          if constexpr (SCATTER) items[at] = make_float4(x, y, z, __uint_as_float(out + uint32_t(j)));
        }
      }
    }
    __syncthreads();
    if constexpr (!SCATTER) {
      for (int c = threadIdx.x; c < ncells; c += kThreads) hr[c] = h[c];
      __syncthreads();
    }
  }
}

// hist[row][cell] of each type's rows to the counts of the rows before it;
// base[type][cell] = the type's count.
__global__ __launch_bounds__(256) void column_kernel(const int32_t *__restrict__ slot_rows, int bits,
                                                     uint32_t *__restrict__ hist, uint32_t *__restrict__ base) {
  const int slot = blockIdx.y, ncells = 1 << bits;
  const int c = int(blockIdx.x) * 256 + int(threadIdx.x);
  if (c >= ncells) return;
  const int r1 = slot_rows[slot + 1];
  uint32_t run = 0;
  int r = slot_rows[slot];
  for (; r + 8 <= r1; r += 8) {  // eight loads in flight
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = hist[size_t(r + k) * size_t(ncells) + size_t(c)];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      hist[size_t(r + k) * size_t(ncells) + size_t(c)] = run;
      run += v[k];
    }
  }
  for (; r < r1; r++) {
    const uint32_t v = hist[size_t(r) * size_t(ncells) + size_t(c)];
    hist[size_t(r) * size_t(ncells) + size_t(c)] = run;
    run += v;
  }
  base[size_t(slot) * size_t(ncells) + size_t(c)] = run;
}

// base[type][cell] from counts to the first item of the cell; one
// work-group per type.
__global__ __launch_bounds__(kThreads) void scan_kernel(const int32_t *__restrict__ slot_items, int bits,
                                                        uint32_t *__restrict__ base) {
  __shared__ uint32_t wsum[kThreads / 64];
  const int per = (1 << bits) >> 10 ? (1 << bits) >> 10 : 1;  // cells per work-item: 4 (12 bits) or 1
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = int(threadIdx.x) * per;
  const bool on = c0 < (1 << bits);
  uint32_t *b = base + (size_t(blockIdx.x) << bits);
  uint32_t v[4], sum = 0;
  for (int i = 0; i < per; i++) {
    v[i] = on ? b[c0 + i] : 0u;
    sum += v[i];
  }
  uint32_t x = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  uint32_t run = uint32_t(slot_items[blockIdx.x]) + x - sum;
  for (int w = 0; w < wave; w++) run += wsum[w];
  if (on)
    for (int i = 0; i < per; i++) {
      b[c0 + i] = run;
      run += v[i];
    }
}

// Points as items (Points::build; 262,144 points of 34 types against 4,096
// atoms, a whole call: 3.45 ms with the points grouped by type on the host
// and every pair scored, 0.76 ms sorted here): the box of them and cleared
// counts, then the counts per (slot, cell), then, the counts having become
// first places, each into its place.
struct PointsIn {
  const float4 *packed;
  const float *xyz;
  const int32_t *slots;
  size_t n;
  __device__ __forceinline__ float4 get(size_t i) const {
    if (packed) return packed[i];
    return make_float4(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], __int_as_float(slots[i]));
  }
};

__global__ __launch_bounds__(kThreads) void point_box_kernel(const PointsIn in, uint32_t *__restrict__ counts,
                                                             size_t ncounts, float *__restrict__ bounds) {
  __shared__ float part[kThreads / 64][6];
  const size_t first = size_t(blockIdx.x) * kThreads + threadIdx.x, step = size_t(gridDim.x) * kThreads;
  for (size_t i = first; i < ncounts; i += step) counts[i] = 0u;
  float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (size_t i = first; i < in.n; i += step) {
    const float4 p = in.get(i);
    v[0] = fminf(v[0], p.x), v[3] = fmaxf(v[3], p.x);
    v[1] = fminf(v[1], p.y), v[4] = fmaxf(v[4], p.y);
    v[2] = fminf(v[2], p.z), v[5] = fmaxf(v[5], p.z);
  }
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const float a = k < 3 ? wave_min(v[k]) : wave_max(v[k]);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][k] = a;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    float a = part[0][threadIdx.x];
    for (int w = 1; w < kThreads / 64; w++)
      a = threadIdx.x < 3 ? fminf(a, part[w][threadIdx.x]) : fmaxf(a, part[w][threadIdx.x]);
    bounds[size_t(blockIdx.x) * 6 + threadIdx.x] = a;
  }
}

template <int SCATTER>
__global__ __launch_bounds__(kThreads) void point_bin_kernel(const PointsIn in, const float *__restrict__ bounds,
                                                             int nbounds, int bits, uint32_t *__restrict__ counts,
                                                             float4 *__restrict__ items) {
  __shared__ uint16_t curve[kCells];
  __shared__ float red[6];
  for (int i = threadIdx.x; i < kCells; i += kThreads) curve[i] = kCurve.place[i];  // (cell_grid waits for it)
  const Space all{{-FLT_MAX, -FLT_MAX, -FLT_MAX}, {FLT_MAX, FLT_MAX, FLT_MAX}, 0.f};
  const CellGrid g = cell_grid(bounds, nbounds, all, red);
  for (size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x; i < in.n; i += size_t(gridDim.x) * kThreads) {
    const float4 p = in.get(i);
    const uint32_t c = cell_of(g, curve, p.x, p.y, p.z) >> (12 - bits);
    const uint32_t at = atomicAdd(&counts[(size_t(__float_as_int(p.w)) << bits) + c], 1u);
    if constexpr (SCATTER) items[at] = make_float4(p.x, p.y, p.z, __uint_as_float(uint32_t(i)));
  }
}

// The protein atoms of `mask` (lanes of the wave's 64 atoms x, y, z), all of
// one group, in order.
template <int RB, int FORM, bool CHG, bool DSLV>
__device__ __forceinline__ void mask_pairs(uint64_t mask, float x, float y, float z, const PairCoef &c,
                                           const float (&lx)[RB], const float (&ly)[RB], const float (&lz)[RB],
                                           float (&e)[RB]) {
  float c0 = 0.f, e0 = 0.f;
  if constexpr (FORM == kFormD) {
    if constexpr (CHG) c0 = vgpr_copy(c.c0);
    if constexpr (DSLV) e0 = vgpr_copy(c.e0);
  }
  do {
    const int j = __builtin_ctzll(mask);
    mask &= mask - 1;
    float4 p;
    p.x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
    p.y = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), j));
    p.z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), j));
    p.w = 0.f;
    atom_pairs<RB, FORM, CHG, DSLV>(p, c, c0, e0, lx, ly, lz, e);
  } while (mask);
}

// The same, each atom with the hinges whose reach it is in only (bits of ms,
// mq, md); the others are exactly zero for all the items (of the 150 atoms per
// item of the 4,096 x 64 deck a fifth are within steric reach, three fifths
// within the charge's, four fifths within the desolvation's: 9.2 VALU of
// arithmetic per pair instead of 11.1).
// The tests are scalar branches between a pair's 6 distance VALU and the 2 of
// each hinge: they pay with four items per lane or more (4,096 x 64 x
// 1,048,576: 5.00 -> 4.46 ms; with one or two the branches cost as much).
template <int RB, int FORM>
__device__ __forceinline__ void mask_hinges(uint64_t mask, uint64_t ms, uint64_t mq, uint64_t md, float x, float y,
                                            float z, const PairCoef &c, const float (&lx)[RB], const float (&ly)[RB],
                                            const float (&lz)[RB], float (&e)[RB]) {
  const float c0 = vgpr_copy(c.c0), e0 = vgpr_copy(c.e0);
  do {
    const int j = __builtin_ctzll(mask);
    mask &= mask - 1;
    const float px = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
    const float py = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), j));
    const float pz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), j));
    float d[RB];
#pragma unroll
    for (int k = 0; k < RB; k++) {
      d[k] = pair_distance(lx[k] - px, ly[k] - py, lz[k] - pz);
      if constexpr (FORM == kFormB) d[k] -= c.radij;
    }
    if (ms >> j & 1)
#pragma unroll
      for (int k = 0; k < RB; k++) e[k] = steric<FORM>(d[k], c, e[k]);
    if (mq >> j & 1)
#pragma unroll
      for (int k = 0; k < RB; k++) e[k] = charge<FORM>(d[k], c, c0, e[k]);
    if (md >> j & 1)
#pragma unroll
      for (int k = 0; k < RB; k++) e[k] = desolvation<FORM>(d[k], c, e0, e[k]);
  } while (mask);
}

// The atoms of a work-group's share of the protein that any of its waves can
// need: list[0 .. n) in order, of atoms base .. base + kShare - 1.
constexpr int kShare = 4096;

// One wave per 64 x RB consecutive items of one type, four waves to a
// work-group.  With LIST (large proteins) the work-group first lists the protein atoms within reach of
// its items' box, 4,096 at a time (each wave tests a quarter, 64 atoms to a
// step); each wave then takes the list, or the protein, 64 atoms at a time
// (lane = atom) against its own items' box, and every atom in reach out of its lane (three
// readlanes) to all lanes' RB items.  RB > 1 shares the steps and the
// readlanes between items at the price of a larger box; VALU issue bounds it
// (11 VALU per pair in reach of the box with eight items per lane, its atom's
// lane reads and the box tests among them).
template <int RB, int FORM, bool LIST>
__global__ __launch_bounds__(256) void score_kernel(const float4 *__restrict__ protein, int natpro,
                                                    const PairCoef *__restrict__ coef,
                                                    const float4 *__restrict__ reach2, int ngroups,
                                                    const float4 *__restrict__ items,
                                                    const int32_t *__restrict__ slot_items,
                                                    const int32_t *__restrict__ slot_units, int nslots, int nunits,
                                                    float scale, float *__restrict__ partial) {
  __shared__ uint16_t list[LIST ? kShare : 1];
  __shared__ float box[4][6];
  __shared__ int count[4], slots[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int unit = int(blockIdx.x) * 4 + wave, u = min(unit, nunits - 1);
  if (!LIST && unit >= nunits) return;  // (with LIST: the last unit again, for its share of the list)
  int slot = 0;  // the last type whose first unit is at or before u
  for (int s0 = 0; s0 < nslots; s0 += 64)
    slot += __popcll(__ballot(s0 + lane < nslots && slot_units[s0 + lane + 1] <= u));
  const int i1 = slot_items[slot + 1];
  const int i0 = slot_items[slot] + (u - slot_units[slot]) * 64 * RB;

  float lx[RB], ly[RB], lz[RB], e[RB], part[RB];
  uint32_t out[RB];
  float bl[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, bh[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
#pragma unroll
  for (int k = 0; k < RB; k++) {
    const float4 it = items[min(i0 + k * 64 + lane, i1 - 1)];  // (past the end: the last item again, not written)
    lx[k] = it.x;
    ly[k] = it.y;
    lz[k] = it.z;
    out[k] = __float_as_uint(it.w);
    e[k] = part[k] = 0.f;
    bl[0] = fminf(bl[0], it.x), bh[0] = fmaxf(bh[0], it.x);
    bl[1] = fminf(bl[1], it.y), bh[1] = fmaxf(bh[1], it.y);
    bl[2] = fminf(bl[2], it.z), bh[2] = fmaxf(bh[2], it.z);
  }
  float wl[3], wh[3];  // the work-group's box
#pragma unroll
  for (int k = 0; k < 3; k++) {
    bl[k] = wave_min(bl[k]);
    bh[k] = wave_max(bh[k]);
    if (LIST && lane == 0) {
      box[wave][k] = bl[k];
      box[wave][3 + k] = bh[k];
    }
  }
  const float4 *rw = reach2;
  if constexpr (LIST) {
    if (lane == 0) slots[wave] = slot;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; k++) {
      wl[k] = fminf(fminf(box[0][k], box[1][k]), fminf(box[2][k], box[3][k]));
      wh[k] = fmaxf(fmaxf(box[0][3 + k], box[1][3 + k]), fmaxf(box[2][3 + k], box[3][3 + k]));
    }
    // the reaches of the work-group's type, or of any type where it has several (the row behind the types')
    const bool one = slots[0] == slots[1] && slots[0] == slots[2] && slots[0] == slots[3];
    rw = reach2 + size_t(__builtin_amdgcn_readfirstlane(one ? slots[0] : nslots)) * size_t(ngroups);
  }
  const float4 *r2 = reach2 + size_t(slot) * size_t(ngroups);
  const PairCoef *cs = coef + size_t(slot) * size_t(ngroups);
  auto at = [&](int i) { return LIST ? int(list[i]) : i; };
  PairCoef c{};
  int cur = -1;
  for (int base = 0; base < natpro; base += kShare) {
    const int n = min(kShare, natpro - base), steps = (n + 63) >> 6;
    int total = n;  // atoms of the share to score against: the listed ones, or all
    if constexpr (LIST) {
      const int s0 = steps * wave >> 2, s1 = steps * (wave + 1) >> 2;  // at most 16 of 64 steps
      uint64_t mine = 0;  // lane i: the mask of step s0 + i
      int found = 0;
      for (int st = s0; st < s1; st++) {
        const int i = st * 64 + lane;
        const float4 p = protein[base + min(i, n - 1)];
        const float dx = p.x - __builtin_amdgcn_fmed3f(p.x, wl[0], wh[0]);
        const float dy = p.y - __builtin_amdgcn_fmed3f(p.y, wl[1], wh[1]);
        const float dz = p.z - __builtin_amdgcn_fmed3f(p.z, wl[2], wh[2]);
        const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
        const uint64_t m = __ballot(i < n && d2 < rw[__float_as_int(p.w)].w);
        if (lane == st - s0) mine = m;
        found += __popcll(m);
      }
      if (lane == 0) count[wave] = found;
      __syncthreads();
      int to = 0;
      for (int w = 0; w < wave; w++) to += count[w];
      total = __builtin_amdgcn_readfirstlane(count[0] + count[1] + count[2] + count[3]);
      for (int st = s0; st < s1; st++) {
        const uint32_t mlo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(mine)), st - s0));
        const uint32_t mhi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(mine >> 32)), st - s0));
        const uint64_t m = uint64_t(mhi) << 32 | mlo;
        if (m >> lane & 1) list[to + __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u))] = uint16_t(st * 64 + lane);
        to += __popcll(m);
      }
      __syncthreads();
    }
    if (total) {
      // two steps ahead: the atoms; one step ahead: their reach
      float4 p = protein[base + at(min(lane, total - 1))], p1 = protein[base + at(min(64 + lane, total - 1))];
      float4 reach = r2[__float_as_int(p.w)];
      for (int k0 = 0; k0 < total; k0 += 64) {
        const float4 reach1 = r2[__float_as_int(p1.w)];
        const float4 p2 = protein[base + at(min(k0 + 128 + lane, total - 1))];
        const float dx = p.x - __builtin_amdgcn_fmed3f(p.x, bl[0], bh[0]);
        const float dy = p.y - __builtin_amdgcn_fmed3f(p.y, bl[1], bh[1]);
        const float dz = p.z - __builtin_amdgcn_fmed3f(p.z, bl[2], bh[2]);
        const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
        const bool on = k0 + lane < total;
        uint64_t mask = __ballot(on && d2 < reach.w), ms = 0, mq = 0, md = 0;
        if constexpr (RB >= 4) {
          ms = __ballot(on && d2 < reach.x);
          mq = __ballot(on && d2 < reach.y);
          md = __ballot(on && d2 < reach.z);
        }
        const int pg = __float_as_int(p.w);
        while (mask) {
          const int g = __builtin_amdgcn_readlane(pg, __builtin_ctzll(mask));
          if (g != cur) {
#pragma unroll
            for (int k = 0; k < RB; k++) {
              e[k] += part[k];
              part[k] = 0.f;
            }
            cur = g;
            c = cs[g];
          }
          const uint64_t sub = mask & __ballot(pg == g);
          mask &= ~sub;
          if constexpr (RB >= 4) {
            mask_hinges<RB, FORM>(sub, ms, mq, md, p.x, p.y, p.z, c, lx, ly, lz, part);
          } else {
            const bool chg = c.wq != 0.f, dslv = c.wd != 0.f;
            if (chg && dslv) mask_pairs<RB, FORM, true, true>(sub, p.x, p.y, p.z, c, lx, ly, lz, part);
            else if (chg) mask_pairs<RB, FORM, true, false>(sub, p.x, p.y, p.z, c, lx, ly, lz, part);
            else if (dslv) mask_pairs<RB, FORM, false, true>(sub, p.x, p.y, p.z, c, lx, ly, lz, part);
            else mask_pairs<RB, FORM, false, false>(sub, p.x, p.y, p.z, c, lx, ly, lz, part);
          }
        }
        p = p1;
        p1 = p2;
        reach = reach1;
      }
    }
    if (LIST && base + kShare < natpro) __syncthreads();  // (the list is rewritten)
  }
  if (unit >= nunits) return;
#pragma unroll
  for (int k = 0; k < RB; k++)
    if (i0 + k * 64 + lane < i1) partial[out[k]] = (e[k] + part[k]) * scale;
}

// p[0] + p[stride] + ... in order, eight loads in flight.
__device__ __forceinline__ float sum_column(const float *__restrict__ p, int n, size_t stride) {
  float e = 0.f;
  int a = 0;
  for (; a + 8 <= n; a += 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = p[size_t(a + k) * stride];
#pragma unroll
    for (int k = 0; k < 8; k++) e += v[k];
  }
  for (; a < n; a++) e += p[size_t(a) * stride];
  return e;
}

// energies[row] = half the sum of the pose's atoms' energies, in the
// ligand's order.  `per` work-groups of 256 per block.
__global__ __launch_bounds__(256) void reduce_kernel(const Block *__restrict__ blocks, int per,
                                                     const float *__restrict__ partial, float *__restrict__ energies) {
  const Block bk = blocks[blockIdx.x / unsigned(per)];
  const int j = int(blockIdx.x % unsigned(per)) * 256 + int(threadIdx.x);
  if (j >= bk.npose) return;
  energies[size_t(bk.pose_off) + size_t(j)] =
      0.5f * sum_column(partial + size_t(bk.part_off) + size_t(j), bk.natlig, bk.part_stride);
}

// Few poses leave a wave per 64 of them alone with every pair: a serial chain
// on a nearly idle device (938 x 26 atoms x 64 poses took 980 us, and takes
// 14; 700 x 19 x 4,096, 574 and 31; latency and the last waves bound it).  One work-group of `blockDim.x / 64` waves per (64 poses, ligand
// atom): its waves share the groups, their parts meet in LDS and wave 0 adds
// them in order (SPLIT); or, where those waves are enough already, one wave
// per (64 poses, ligand atom).  out[atom][pose], rows of 64 poses per tile.
template <int FORM, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 1024 : 256) void direct_kernel(
    const float4 *__restrict__ protein, const int32_t *__restrict__ group_begin, const PairCoef *__restrict__ coef,
    const float4 *__restrict__ ligand, const float *__restrict__ poses, size_t stride, size_t n, int ntiles,
    int natlig, int ngroups, const int32_t *__restrict__ skip, float *__restrict__ out) {
  extern __shared__ float parts[];  // SPLIT: [ngroups][64]
  if (skip && *skip) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int nwaves = int(blockDim.x >> 6);
  const int64_t w = SPLIT ? int64_t(blockIdx.x) : int64_t(blockIdx.x) * nwaves + wave;
  const int il = int(w / ntiles), tile = int(w - int64_t(il) * ntiles);
  if (il >= natlig) return;  // (whole waves; with SPLIT none)
  const size_t j = size_t(tile) * 64 + size_t(lane);
  const Xform t = make_xform(poses, stride, j < n ? j : n - 1);
  const float4 la = ligand[il];
  const float lx[1] = {place(t.m[0], t.m[1], t.m[2], t.m[3], la)};
  const float ly[1] = {place(t.m[4], t.m[5], t.m[6], t.m[7], la)};
  const float lz[1] = {place(t.m[8], t.m[9], t.m[10], t.m[11], la)};
  const PairCoef *cl = coef + size_t(il) * size_t(ngroups);
  float e[1] = {0.f};
  if constexpr (SPLIT) {
    for (int g = wave; g < ngroups; g += nwaves) {
      e[0] = 0.f;
      group_dispatch<1, FORM>(protein, group_begin[g], group_begin[g + 1], cl[g], lx, ly, lz, e);
      parts[g * 64 + lane] = e[0];
    }
    __syncthreads();
    if (wave) return;
    e[0] = 0.f;
#pragma unroll 8
    for (int g = 0; g < ngroups; g++) e[0] += parts[g * 64 + lane];
  } else {
    for (int g = 0; g < ngroups; ++g)
      group_dispatch<1, FORM>(protein, group_begin[g], group_begin[g + 1], cl[g], lx, ly, lz, e);
  }
  out[size_t(il) * size_t(ntiles) * 64 + j] = e[0];
}

// Pose energies from the atoms' (partial[atom][pose]), one work-item per pose.
__global__ __launch_bounds__(256) void atom_sum_kernel(const float *__restrict__ partial, size_t npad, size_t n,
                                                       int natlig, const int32_t *__restrict__ skip,
                                                       float *__restrict__ energies) {
  if (skip && *skip) return;
  const size_t j = size_t(blockIdx.x) * 256 + threadIdx.x;
  if (j >= n) return;
  energies[j] = 0.5f * sum_column(partial + j, natlig, npad);
}

template <int PPT, int SCATTER, class... A> void launch_bin(int ntasks, hipStream_t s, A... args) {
  hipLaunchKernelGGL(HIP_KERNEL_NAME(bin_kernel<PPT, SCATTER>), dim3(unsigned(ntasks)), dim3(kThreads), 0, s, args...);
}

template <int SCATTER, class... A> void launch_bin_ppt(int ppt, int ntasks, hipStream_t s, A... args) {
  if (ppt >= 8) launch_bin<8, SCATTER>(ntasks, s, args...);
  else if (ppt >= 4) launch_bin<4, SCATTER>(ntasks, s, args...);
  else if (ppt >= 2) launch_bin<2, SCATTER>(ntasks, s, args...);
  else launch_bin<1, SCATTER>(ntasks, s, args...);
}

template <int RB, int FORM, class... A> void launch_score(bool listed, int nunits, hipStream_t s, A... args) {
  const dim3 grid(unsigned((nunits + 3) / 4));
  if (listed) hipLaunchKernelGGL(HIP_KERNEL_NAME(score_kernel<RB, FORM, true>), grid, dim3(256), 0, s, args...);
  else hipLaunchKernelGGL(HIP_KERNEL_NAME(score_kernel<RB, FORM, false>), grid, dim3(256), 0, s, args...);
}

template <int FORM, class... A> void launch_score_rb(int rb, bool listed, int nunits, hipStream_t s, A... args) {
  if (rb >= 8) launch_score<8, FORM>(listed, nunits, s, args...);
  else if (rb >= 4) launch_score<4, FORM>(listed, nunits, s, args...);
  else if (rb >= 2) launch_score<2, FORM>(listed, nunits, s, args...);
  else launch_score<1, FORM>(listed, nunits, s, args...);
}

constexpr size_t kDirectWaves = 16384;

// Work-groups of the point kernels, for n points.
unsigned point_groups(size_t n) { return unsigned(std::min<size_t>(kMaxBounds, (n + kThreads - 1) / kThreads)); }

// Items per lane for `mean` items of a type: more share the protein's steps,
// fewer keep the box small where items are sparse.  Whole passes at 1, 2, 4
// and 8: 24 k items of a type 73, 78, 98, 128 us; 95 k 340, 315, 317, 450;
// 560 k 2,050, 1,580, 1,330, 1,380; 2.2 M 7,980, 5,980, 4,720, 4,450.
int items_per_lane(int64_t mean) { return mean >= 1100000 ? 8 : mean >= 230000 ? 4 : mean >= 48000 ? 2 : 1; }

// Proteins from which the score kernel lists a work-group's atoms first: with
// and without, 4,096 x 64 x 262,144 1,250 and 1,340 us, 4,096 x 26 x 65,536
// 300 and 316; 938 x 64 x 262,144 617 and 596, 300 x 64 x 131,072 249 and 234
// (15 and 5 steps of 64 atoms per wave are no work worth sharing).
constexpr int kListFrom = 1500;

void score_items(const Scene &sc, int rb, const float4 *items, const int32_t *slot_items, const int32_t *slot_units,
                 int nslots, int nunits, float scale, float *out, hipStream_t s) {
  auto score = [&](auto run) {
    run(rb, sc.natpro >= kListFrom, nunits, s, sc.protein, sc.natpro, sc.coef, sc.reach2, sc.ngroups, items,
        slot_items, slot_units, nslots, nunits, scale, out);
  };
  if (sc.form == kFormD) score([](auto... args) { launch_score_rb<kFormD>(args...); });
  else score([](auto... args) { launch_score_rb<kFormB>(args...); });
}

// Items of one chunk.  Each takes 20 bytes of scratch, its counts up to 16 more
// (Plan::build), and a pose's transform 48.
constexpr int64_t kChunkItems = int64_t(1) << 26;

// The device hands work-group i to XCD i mod 8, each with an L2 of its own.
// Give an XCD a contiguous eighth of the blocks, and all of a type's rows
// before the next type's, so that neighbouring places of a cell are written
// by one XCD at about the same time and leave its L2 as fewer partial lines
// (938 x 26 x 65,536: 136 -> 127 us a pass; 4,096 x 64 x 1,048,576: 4.45 ->
// 4.34 ms).
void spread_tasks(std::vector<Task> &tasks, const std::vector<int32_t> &refs, const std::vector<Row> &rows,
                  size_t nblocks) {
  constexpr size_t kXcds = 8;
  auto slot = [&](const Task &t) { return rows[size_t(refs[size_t(t.ref0)])].slot; };
  std::stable_sort(tasks.begin(), tasks.end(), [&](const Task &a, const Task &b) { return slot(a) < slot(b); });
  std::vector<std::vector<Task>> of(kXcds);
  for (const Task &t : tasks) of[size_t(t.block) * kXcds / nblocks].push_back(t);
  tasks.clear();
  for (size_t k = 0, more = 1; more; k++) {
    more = 0;
    for (const std::vector<Task> &x : of)
      if (k < x.size()) {
        tasks.push_back(x[k]);
        more = 1;
      }
  }
}

int slot_of(const float4 &a) {
  int s;
  std::memcpy(&s, &a.w, sizeof s);
  return s;
}

}  // namespace

bool pair_reach(const PairCoef &c, float r[3]) {
  const float all[] = {c.radij, c.neg_rr, c.neg_e1, c.wq, c.neg_rd, c.wd, c.c0, c.e0};
  for (float v : all)
    if (!std::isfinite(v)) return false;
  if (!(c.radij > 0.f) || !(c.neg_rr < 0.f) || !(c.neg_e1 < 0.f) || (c.wd != 0.f && !(c.neg_rd < 0.f))) return false;
  auto wide = [](float a, float b) { return std::max(a, b) * 1.0001f + 1e-3f; };
  r[0] = wide(c.radij, -1.0f / c.neg_rr);
  r[1] = c.wq != 0.f ? wide(c.c0 / -c.neg_e1, c.radij - 1.0f / c.neg_e1) : -1.f;
  r[2] = c.wd != 0.f ? wide(c.e0 / -c.neg_rd, c.radij - 1.0f / c.neg_rd) : -1.f;
  for (int k = 0; k < 3; k++)
    if (!std::isfinite(r[k] * r[k])) return false;
  return true;
}

bool reach_table(const std::vector<PairCoef> &coef, size_t ngroups, std::vector<float4> &reach2, float *largest) {
  reach2.resize(coef.size() + ngroups);  // (the last row: the largest reaches of any slot)
  for (size_t g = 0; g < ngroups; g++) reach2[coef.size() + g] = make_float4(-1.f, -1.f, -1.f, 0.f);
  *largest = 0.f;
  for (size_t i = 0; i < coef.size(); i++) {
    float r[3];
    if (!pair_reach(coef[i], r)) return false;
    const float most = std::max({r[0], r[1], r[2]});
    *largest = std::max(*largest, most);
    auto square = [](float v) { return v < 0.f ? -1.f : v * v; };
    reach2[i] = make_float4(square(r[0]), square(r[1]), square(r[2]), square(most));
    float4 &any = reach2[coef.size() + i % ngroups];
    any.w = std::max(any.w, square(most));
  }
  return true;
}

void protein_box(const std::vector<float> &xyzw, float reach, float lo[3], float hi[3]) {
  for (int k = 0; k < 3; k++) {
    float a = FLT_MAX, b = -FLT_MAX;
    for (size_t i = size_t(k); i < xyzw.size(); i += 4)
      if (std::isfinite(xyzw[i])) {
        a = std::min(a, xyzw[i]);
        b = std::max(b, xyzw[i]);
      }
    lo[k] = a - reach;
    hi[k] = b + reach;
  }
}

namespace {

// Estimates of a pass in microseconds beyond a launch and its wait, for the
// choice between the forms; ps per item and pose.  Measured over proteins of
// 1 to 4,096 atoms (1 to 34 groups), ligands of 1 to 500, 65,536 to 4 M poses.
//
// Tiled: 64 x 64 atoms x 1,048,576 poses 34, 25, 25 and 28 ps an item with 1,
// 2, 4 and 8 poses a register block, 16 x 64 13, 8.2, 7.4 and 7.7, 1 x 64 1.7
// to 1.1, 4,096 x 26 1,207; a group costs the more the fewer atoms it has and
// poses share it.  With w waves per SIMD it takes 1 + 2.3 / (sqrt(rb) w^1.5)
// times as long (64 x 64 with rb 1: 3.9 at w = 1, 1.31 at 4).  The persistent
// kernel takes a pose's transform and its place in the queue worse: 256 x 20 x
// 4,096 poses against one atom 265 us with rb 1, 131 with 4.
double tiled_us(const Work &w, int ppwi, int rb, double pose_ps = kPlainPose) {
  const double natpro = double(w.natpro), groups = double(w.ngroups) * std::min(1.0, 64.0 / natpro);
  const double full = w.items * (0.29 * natpro + groups * (0.1 + 0.4 / rb)) + pose_ps * w.poses;
  return full * 1e-6 * (1.0 + 2.3 / std::sqrt(double(rb)) * std::pow(65536.0 * ppwi / w.poses, 1.5));
}

// Sorted, small proteins: 30 ps an item however few the atoms (1 x 64 x
// 1,048,576 26, 64 x 64 and 128 x 64 29.9), 58 where a pose has one.
double sorted_us(const Work &w) {
  return 30.0 + (w.items * (29.5 + 0.008 * double(w.natpro)) + 29.0 * w.poses) * 1e-6;
}

// Direct: 5 ps an item (1 x 64 x 262,144), 15.7 (16 x 8), 42 (64 x 8), and a
// second launch.
double direct_us(const Work &w) {
  const double natpro = double(w.natpro);
  const double item = 0.305 * natpro + (4.0 + 0.55 * double(w.ngroups)) * std::min(1.0, 64.0 / natpro);
  return 6.0 + (w.items * item + 12.0 * w.poses) * 1e-6;
}

}  // namespace

bool worth_sorting(const Work &w, int ppwi, int rb, double pose_ps) {
  // Against the direct pass: that scores some 1.8e9 pairs a millisecond; the sort's seven
  // launches cost 40-50 us whatever the size, and with few items (large
  // boxes) scoring them grows with the protein.  Both measured, direct and
  // sorted, over 64 .. 131,072 poses: 300 x 8 atoms cross at 1.5e8 pairs
  // (67 and 65 us), 700 x 19 at 1e8, 938 x 26 at 1.4e8, 938 x 64 at 2e8,
  // 4,096 x 26 at 4.4e8 (189 and 192 us), 4,096 x 96 at 6e8.  A segment is to
  // fill the work-groups that sort it.
  // Against a tiled kernel: sorting moves some 30 bytes an item, which costs
  // more than the few pairs of a small protein (64 x 64 x 1,048,576: 2,000 us,
  // 1,690 tiled with two poses per work-item; 4 x 64 x 262,144: 504 and 91).
  const double natpro = double(w.natpro);
  return w.items * natpro >= 6e7 + 8e4 * natpro && w.items >= 4096.0 * double(w.nsegs) &&
         sorted_us(w) <= tiled_us(w, ppwi, rb, pose_ps);
}

bool worth_direct(const Work &w, int ppwi, int rb, size_t passes, double wait_us) {
  // 1 x 64 x 262,144: 102 us, 44 tiled with two poses per work-item; 64 x 8 x
  // 262,144: 107 and 105; larger proteins: nothing between them where the
  // tiled kernel has the poses to fill the device, else the direct pass.  A
  // tenth is within the estimates.  Split into many launches (3 us each) the
  // direct pass loses to a full tiled kernel: 64 x 64 x 1,048,576 in 65
  // launches 3,090 us, 1,810 tiled; 300 x 64 7,110 and 6,480.
  const bool large = w.natpro >= 128;
  if (large && passes == 1) return true;
  return direct_us(w) + 3.0 * double(passes - 1) <= (large ? 1.0 : 1.15) * tiled_us(w, ppwi, rb) + wait_us;
}

int Plan::build(const std::vector<float4> &atoms, const std::vector<int32_t> &lig_off, int nslots,
                const std::vector<Segment> &segs) {
  chunks_.clear();
  nslots_ = nslots;
  nsegs_ = segs.size();
  items_ = poses_ = 0;
  radius_ = 0.f;
  // every ligand's atoms grouped by type (stable), w bits: place in the ligand
  const size_t nlig = lig_off.size() - 1;
  std::vector<float4> grouped;
  std::vector<std::vector<Row>> lig_rows(nlig);
  for (size_t l = 0; l < nlig; l++) {
    const int32_t a0 = lig_off[l], n = lig_off[l + 1] - a0;
    std::vector<int32_t> order(static_cast<size_t>(n), 0);
    for (int32_t i = 0; i < n; i++) order[size_t(i)] = i;
    std::stable_sort(order.begin(), order.end(),
                     [&](int32_t x, int32_t y) { return slot_of(atoms[size_t(a0 + x)]) < slot_of(atoms[size_t(a0 + y)]); });
    for (int32_t i : order) {
      float4 a = atoms[size_t(a0 + i)];
      const int s = slot_of(a);
      const float r = std::sqrt(a.x * a.x + a.y * a.y + a.z * a.z);
      if (std::isfinite(r)) radius_ = std::max(radius_, r);
      if (lig_rows[l].empty() || lig_rows[l].back().slot != s)
        lig_rows[l].push_back(Row{0, int32_t(grouped.size()), 0, s});
      lig_rows[l].back().natoms++;
      std::memcpy(&a.w, &i, sizeof i);
      grouped.push_back(a);
    }
  }
  radius_ = radius_ * 1.0001f;

  // pieces of segments, in chunks of at most kChunkItems items
  struct Piece {
    int32_t lig;
    int64_t seg_off, first, n;
  };
  std::vector<std::vector<Piece>> parts(1);
  int64_t room = kChunkItems;
  for (const Segment &s : segs) {
    const int64_t L = lig_off[size_t(s.lig) + 1] - lig_off[size_t(s.lig)];
    if (L <= 0 || L > kChunkItems / 64) return BUDE_OK;
    items_ += double(L) * double(s.n);
    poses_ += double(s.n);
    for (int64_t j = 0; j < s.n;) {
      int64_t take = std::min(s.n - j, room / L);
      if (take < s.n - j) take = take / 64 * 64;
      if (take <= 0) {
        parts.emplace_back();
        room = kChunkItems;
        continue;
      }
      parts.back().push_back(Piece{s.lig, s.pose_off, j, take});
      room -= take * L;
      j += take;
    }
  }
  if (parts.back().empty()) parts.pop_back();

  std::vector<char> bytes;
  auto put = [&](const void *p, size_t n) {
    bytes.resize((bytes.size() + 63) / 64 * 64);
    const size_t at = bytes.size();
    bytes.insert(bytes.end(), static_cast<const char *>(p), static_cast<const char *>(p) + n);
    return at;
  };
  for (const std::vector<Piece> &pieces : parts) {
    Chunk ch{};
    // poses per work-item: as many as leave enough (type, block) rows to fill the device
    int64_t nrows = 0, nitems = 0, longest = 0;
    for (const Piece &p : pieces) longest = std::max(longest, p.n);
    for (ch.ppt = 8;; ch.ppt /= 2) {
      if (ch.ppt > 1 && kThreads * ch.ppt / 2 >= longest) continue;
      nrows = 0;
      for (const Piece &p : pieces)
        nrows += (p.n + kThreads * ch.ppt - 1) / (kThreads * ch.ppt) * int64_t(lig_rows[size_t(p.lig)].size());
      if (ch.ppt == 1 || nrows >= 512) break;
    }
    std::vector<Block> blocks;
    std::vector<std::vector<Row>> by_slot(static_cast<size_t>(nslots));
    std::vector<int32_t> slot_rows(size_t(nslots) + 1, 0), slot_items(size_t(nslots) + 1, 0),
        slot_units(size_t(nslots) + 1, 0);
    std::vector<int64_t> count(static_cast<size_t>(nslots), 0);
    int64_t part = 0, xf = 0;
    for (const Piece &p : pieces) {
      const int64_t L = lig_off[size_t(p.lig) + 1] - lig_off[size_t(p.lig)];
      for (int64_t j = 0; j < p.n; j += kThreads * ch.ppt) {
        const int64_t n = std::min<int64_t>(kThreads * ch.ppt, p.n - j);
        for (Row r : lig_rows[size_t(p.lig)]) {
          r.block = int32_t(blocks.size());
          by_slot[size_t(r.slot)].push_back(r);
          count[size_t(r.slot)] += n * r.natoms;
        }
        blocks.push_back(Block{p.seg_off + p.first + j, uint32_t(part + j), uint32_t(p.n), int32_t(n), int32_t(L),
                               uint32_t(xf + j), int32_t(p.first + j)});
      }
      part += p.n * L;
      xf += p.n;
    }
    int64_t used = 0;
    for (int t = 0; t < nslots; t++) {
      nitems += count[size_t(t)];
      used += count[size_t(t)] > 0;
    }
    const int64_t mean = nitems / std::max<int64_t>(1, used);
    ch.rb = items_per_lane(mean);
    ch.cell_bits = mean >= 16384 ? 12 : 9;
    // Short segments have many rows of few items: no more than four counts an
    // item, so that the counts stay a part of the scratch (2,048 ligands of 64
    // atoms x 64 poses against 300 atoms: 1,244 MB and 1,480 us a pass with 12
    // bits, 432 and 590 with 9; 256 of 52 x 256 against 4,096: 198 MB and 502
    // us, 100 and 504; one count an item costs 730 there, the cells too coarse).
    while (ch.cell_bits > 0 && nrows << ch.cell_bits > 4 * nitems) ch.cell_bits -= 3;
    std::vector<Row> rows;
    std::vector<std::vector<int32_t>> refs_of(blocks.size());
    for (int t = 0; t < nslots; t++) {
      for (const Row &r : by_slot[size_t(t)]) {
        refs_of[size_t(r.block)].push_back(int32_t(rows.size()));
        rows.push_back(r);
      }
      slot_rows[size_t(t) + 1] = int32_t(rows.size());
      slot_items[size_t(t) + 1] = slot_items[size_t(t)] + int32_t(count[size_t(t)]);
      slot_units[size_t(t) + 1] =
          slot_units[size_t(t)] + int32_t((count[size_t(t)] + 64 * ch.rb - 1) / (64 * ch.rb));
    }
    const size_t per_task = std::max<size_t>(1, rows.size() / 768);
    std::vector<int32_t> refs;
    std::vector<Task> tasks;
    for (size_t b = 0; b < blocks.size(); b++)
      for (size_t i = 0; i < refs_of[b].size(); i += per_task) {
        const size_t n = std::min(per_task, refs_of[b].size() - i);
        tasks.push_back(Task{int32_t(b), int32_t(refs.size()), int32_t(n), 0});
        refs.insert(refs.end(), refs_of[b].begin() + long(i), refs_of[b].begin() + long(i + n));
      }
    spread_tasks(tasks, refs, rows, blocks.size());
    ch.nblocks = int(blocks.size());
    ch.ntasks = int(tasks.size());
    ch.nrows = uint32_t(rows.size());
    ch.nitems = uint32_t(nitems);
    ch.npartial = uint32_t(part);
    ch.nxform = uint32_t(xf);
    ch.nunits = slot_units.back();
    ch.blocks = put(blocks.data(), blocks.size() * sizeof(Block));
    ch.tasks = put(tasks.data(), tasks.size() * sizeof(Task));
    ch.refs = put(refs.data(), refs.size() * 4);
    ch.rows = put(rows.data(), rows.size() * sizeof(Row));
    ch.slot_rows = put(slot_rows.data(), slot_rows.size() * 4);
    ch.slot_items = put(slot_items.data(), slot_items.size() * 4);
    ch.slot_units = put(slot_units.data(), slot_units.size() * 4);
    chunks_.push_back(ch);
  }
  int st = atoms_.assign(grouped.data(), grouped.size() * sizeof(float4));
  if (!st) st = tables_.assign(bytes.data(), bytes.size());
  if (st == BUDE_ERR_OUT_OF_MEMORY) {
    chunks_.clear();
    st = BUDE_OK;
  }
  return st;
}

std::array<size_t, 7> Plan::layout() const {
  std::array<size_t, 6> n{};
  for (const Chunk &c : chunks_) {
    n[0] = std::max(n[0], size_t(c.nitems) * sizeof(float4));
    n[1] = std::max(n[1], size_t(c.npartial) * sizeof(float));
    n[2] = std::max(n[2], size_t(c.nxform) * 3 * sizeof(float4));
    n[3] = std::max(n[3], (size_t(c.nrows) << c.cell_bits) * sizeof(uint32_t));
    n[4] = std::max(n[4], (size_t(nslots_) << c.cell_bits) * sizeof(uint32_t));
  }
  n[5] = kMaxBounds * 6 * sizeof(float);
  std::array<size_t, 7> at{};
  for (size_t i = 0; i < 6; i++) at[i + 1] = at[i] + ((n[i] + 255) & ~size_t(255));
  return at;
}

int Plan::reserve(Workspace &w) const {
  const size_t old = w.buf.bytes;
  const int st = w.buf.reserve(layout()[6]);
  if (st == BUDE_ERR_OUT_OF_MEMORY && old) (void)w.buf.alloc(old);  // (other plans' passes go on with it)
  return st;
}

hipError_t Plan::launch(const Scene &sc, const Workspace &w, const float *poses, size_t stride, const uint32_t *index,
                        float *energies, hipStream_t s) const {
  if (chunks_.empty() || !fits(w)) return hipErrorInvalidValue;
  Space sp{};
  for (int k = 0; k < 3; k++) {
    sp.lo[k] = sc.lo[k];
    sp.hi[k] = sc.hi[k];
  }
  sp.radius = radius_;
  const auto *tables = static_cast<const char *>(tables_.ptr);
  const auto *atoms = static_cast<const float4 *>(atoms_.ptr);
  const std::array<size_t, 7> at = layout();
  auto *scratch = static_cast<char *>(w.buf.ptr);
  auto *items = reinterpret_cast<float4 *>(scratch + at[0]);
  auto *partial = reinterpret_cast<float *>(scratch + at[1]);
  auto *xf = reinterpret_cast<float4 *>(scratch + at[2]);
  auto *hist = reinterpret_cast<uint32_t *>(scratch + at[3]);
  auto *base = reinterpret_cast<uint32_t *>(scratch + at[4]);
  auto *bounds = reinterpret_cast<float *>(scratch + at[5]);
  for (const Chunk &c : chunks_) {
    const auto *blocks = reinterpret_cast<const Block *>(tables + c.blocks);
    const auto *tasks = reinterpret_cast<const Task *>(tables + c.tasks);
    const auto *refs = reinterpret_cast<const int32_t *>(tables + c.refs);
    const auto *rows = reinterpret_cast<const Row *>(tables + c.rows);
    const auto *slot_rows = reinterpret_cast<const int32_t *>(tables + c.slot_rows);
    const auto *slot_items = reinterpret_cast<const int32_t *>(tables + c.slot_items);
    const auto *slot_units = reinterpret_cast<const int32_t *>(tables + c.slot_units);
    const int nb = std::min(c.nblocks, kMaxBounds);
    hipLaunchKernelGGL(prep_kernel, dim3(unsigned(nb)), dim3(kThreads), 0, s, blocks, c.nblocks, poses, stride, index,
                       xf, size_t(c.nxform), bounds);
    launch_bin_ppt<0>(c.ppt, c.ntasks, s, tasks, blocks, refs, rows, atoms, static_cast<const float4 *>(xf),
                      size_t(c.nxform), static_cast<const float *>(bounds), nb, sp, c.cell_bits, hist,
                      static_cast<const uint32_t *>(base), items);
    hipLaunchKernelGGL(column_kernel, dim3(((1u << c.cell_bits) + 255u) / 256u, unsigned(nslots_)), dim3(256), 0, s, slot_rows,
                       c.cell_bits, hist, base);
    hipLaunchKernelGGL(scan_kernel, dim3(unsigned(nslots_)), dim3(kThreads), 0, s, slot_items, c.cell_bits, base);
    launch_bin_ppt<1>(c.ppt, c.ntasks, s, tasks, blocks, refs, rows, atoms, static_cast<const float4 *>(xf),
                      size_t(c.nxform), static_cast<const float *>(bounds), nb, sp, c.cell_bits, hist,
                      static_cast<const uint32_t *>(base), items);
    score_items(sc, c.rb, items, slot_items, slot_units, nslots_, c.nunits, 1.0f, partial, s);
    const int per = 4 * c.ppt;  // work-groups of 256 per block of 1024 ppt poses
    hipLaunchKernelGGL(reduce_kernel, dim3(unsigned(c.nblocks) * unsigned(per)), dim3(256), 0, s, blocks, per,
                       static_cast<const float *>(partial), energies);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  return hipSuccess;
}

int Points::build(const float4 *packed, const float *xyz, const int32_t *slots, size_t n,
                  const std::vector<size_t> &slot_count, hipStream_t s) {
  if (n == 0 || n > 0x7fffffffu || slot_count.empty())
    return fail(BUDE_ERR_INVALID_ARGUMENT, "points: none, or more than 2^31");
  nslots_ = int(slot_count.size());
  const int64_t mean = int64_t(n / slot_count.size());
  const int bits = mean >= 16384 ? 12 : mean >= 512 ? 9 : 6;
  rb_ = items_per_lane(mean);
  std::vector<int32_t> table(2 * (size_t(nslots_) + 1), 0);
  int32_t *first = table.data(), *unit = first + nslots_ + 1;
  for (int t = 0; t < nslots_; t++) {
    first[t + 1] = first[t] + int32_t(slot_count[size_t(t)]);
    unit[t + 1] = unit[t] + int32_t((int64_t(slot_count[size_t(t)]) + 64 * rb_ - 1) / (64 * rb_));
  }
  if (size_t(first[nslots_]) != n) return fail(BUDE_ERR_INVALID_ARGUMENT, "points: counts do not add up");
  nunits_ = unit[nslots_];
  // one allocation: items, counts, bounds, the table
  auto pad = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t ncounts = size_t(nslots_) << bits;
  const size_t at_counts = pad(n * sizeof(float4)), at_bounds = at_counts + pad(ncounts * 4),
               at_table = at_bounds + pad(kMaxBounds * 24);
  if (int st = buf_.reserve(at_table + table.size() * 4)) return st;
  auto *base = static_cast<char *>(buf_.ptr);
  auto *items = reinterpret_cast<float4 *>(base);
  auto *counts = reinterpret_cast<uint32_t *>(base + at_counts);
  auto *bounds = reinterpret_cast<float *>(base + at_bounds);
  items_ = items;
  slot_items_ = reinterpret_cast<const int32_t *>(base + at_table);
  slot_units_ = slot_items_ + nslots_ + 1;
  if (int st = hip_check(hipMemcpyAsync(base + at_table, table.data(), table.size() * 4, hipMemcpyHostToDevice, s),
                         "hipMemcpyAsync"))
    return st;
  if (int st = hip_check(hipStreamSynchronize(s), "hipStreamSynchronize")) return st;  // (the table is a local)
  const PointsIn in{packed, xyz, slots, n};
  const unsigned groups = point_groups(n);
  hipLaunchKernelGGL(point_box_kernel, dim3(groups), dim3(kThreads), 0, s, in, counts, ncounts, bounds);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(point_bin_kernel<0>), dim3(groups), dim3(kThreads), 0, s, in,
                     static_cast<const float *>(bounds), int(groups), bits, counts, items);
  hipLaunchKernelGGL(scan_kernel, dim3(unsigned(nslots_)), dim3(kThreads), 0, s, slot_items_, bits, counts);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(point_bin_kernel<1>), dim3(groups), dim3(kThreads), 0, s, in,
                     static_cast<const float *>(bounds), int(groups), bits, counts, items);
  return hip_check(hipGetLastError(), "sort points");
}

hipError_t Points::launch(const Scene &sc, float *out, hipStream_t s) const {
  if (!items_) return hipErrorInvalidValue;
  score_items(sc, rb_, items_, slot_items_, slot_units_, nslots_, nunits_, 0.5f, out, s);
  return hipGetLastError();
}

size_t direct_bytes(size_t n, size_t natlig) { return (n + 63) / 64 * 64 * natlig * sizeof(float); }

hipError_t launch_direct(const DirectArgs &a, hipStream_t s) {
  const size_t ntiles = (a.nposes + 63) / 64, npad = ntiles * 64, natlig = size_t(a.natlig);
  if (a.nposes == 0 || ntiles * natlig > 0x7fffffffu || !a.scratch) return hipErrorInvalidValue;
  // waves per (tile, ligand atom): until they number some sixteen per SIMD
  // (256 CUs of 4), so that the last ones end together (4,096 x 26 atoms,
  // 4,096 poses: 198 us with four per SIMD, 152 with sixteen; 938 x 26: 64
  // and 52 us); as far as the parts fit 64 KB of LDS
  size_t split = std::min({size_t(16), size_t(a.ngroups), kDirectWaves / (ntiles * natlig)});
  const size_t lds = size_t(a.ngroups) * 64 * sizeof(float);
  if (lds > 65536) split = 1;
  auto run = [&](auto kernel, size_t blocks, size_t threads, size_t bytes) {
    hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(unsigned(threads)), unsigned(bytes), s, a.protein,
                       a.group_begin, a.coef, a.ligand, a.poses, a.stride, a.nposes, int(ntiles), a.natlig, a.ngroups,
                       a.skip, a.scratch);
  };
  if (split > 1) {
    if (a.form == kFormD) run(direct_kernel<kFormD, true>, ntiles * natlig, 64 * split, lds);
    else run(direct_kernel<kFormB, true>, ntiles * natlig, 64 * split, lds);
  } else {
    if (a.form == kFormD) run(direct_kernel<kFormD, false>, (ntiles * natlig + 3) / 4, 256, 0);
    else run(direct_kernel<kFormB, false>, (ntiles * natlig + 3) / 4, 256, 0);
  }
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  hipLaunchKernelGGL(atom_sum_kernel, dim3(unsigned((a.nposes + 255) / 256)), dim3(256), 0, s, a.scratch, npad,
                     a.nposes, a.natlig, a.skip, a.energies);
  return hipGetLastError();
}

int Deck::prepare(const ProteinGroups &groups, const BudeFFParams *ff, const std::vector<BudeAtom> &atoms,
                  const std::vector<int32_t> &lig_off, const std::vector<Segment> &segs) {
  usable_ = false;
  bool ok = false;
  const int st = plan(groups, ff, atoms, lig_off, segs, &ok);
  if (st || !ok) release();
  usable_ = st == BUDE_OK && ok;
  return st == BUDE_ERR_OUT_OF_MEMORY ? BUDE_OK : st;  // (the tiled kernels need none of it)
}

void Deck::release() {
  usable_ = false;
  plan_.clear();
  for (DeviceBuffer *b : {&work_.buf, &coef_, &reach2_}) b->reset();
}

int Deck::plan(const ProteinGroups &groups, const BudeFFParams *ff, const std::vector<BudeAtom> &atoms,
               const std::vector<int32_t> &lig_off, const std::vector<Segment> &segs, bool *ok) {
  const size_t natpro = size_t(groups.begin.back());
  shape_ = Work{natpro, groups.ngroups(), segs.size()};
  for (const Segment &s : segs) {
    shape_.items += double(lig_off[size_t(s.lig) + 1] - lig_off[size_t(s.lig)]) * double(s.n);
    shape_.poses += double(s.n);
  }
  if (!worth_sorting(shape_, 1, 1, persistent_pose(1)) && !worth_sorting(shape_, 8, 8)) return BUDE_OK;
  // slots: the forcefield types the ligands use, ascending
  std::vector<int32_t> types;
  for (const BudeAtom &a : atoms) types.push_back(a.type);
  std::sort(types.begin(), types.end());
  types.erase(std::unique(types.begin(), types.end()), types.end());
  std::vector<BudeAtom> probe;
  for (int32_t t : types) probe.push_back(BudeAtom{0.f, 0.f, 0.f, t});
  const std::vector<PairCoef> coef = coef_table(probe.data(), probe.size(), groups, ff);
  std::vector<float4> reach2;
  float largest = 0.f;
  if (!reach_table(coef, groups.ngroups(), reach2, &largest)) return BUDE_OK;
  std::vector<float4> slotted;
  for (const BudeAtom &a : atoms) {
    const int32_t s = int32_t(std::lower_bound(types.begin(), types.end(), a.type) - types.begin());
    float4 v = make_float4(a.x, a.y, a.z, 0.f);
    std::memcpy(&v.w, &s, sizeof s);
    slotted.push_back(v);
  }
  if (int st = coef_.upload(coef.data(), coef.size() * sizeof(PairCoef))) return st;
  if (int st = reach2_.upload(reach2.data(), reach2.size() * sizeof(float4))) return st;
  if (int st = plan_.build(slotted, lig_off, int(types.size()), segs)) return st;
  if (plan_.empty()) return BUDE_OK;
  scene_.coef = static_cast<const PairCoef *>(coef_.ptr);
  scene_.reach2 = static_cast<const float4 *>(reach2_.ptr);
  scene_.natpro = int(natpro);
  scene_.ngroups = int(groups.ngroups());
  scene_.form = plain_form();
  protein_box(groups.xyzw, largest, scene_.lo, scene_.hi);
  if (int st = plan_.reserve(work_)) return st;
  *ok = true;
  return BUDE_OK;
}

hipError_t Deck::launch(const float4 *protein, const float *poses, size_t stride, const uint32_t *index,
                        float *energies, hipStream_t s) const {
  if (!usable_) return hipErrorInvalidValue;
  Scene sc = scene_;
  sc.protein = protein;
  return plan_.launch(sc, work_, poses, stride, index, energies, s);
}

}  // namespace items
}  // namespace bude
