// items.h -- exact pose energies from sorted (pose, ligand atom) items.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <vector>

#include "bude_internal.h"
#include "hip_util.h"

namespace bude {
namespace items {

// What the items are scored against: the grouped protein (a group index in
// the w bits of every atom), and per ligand-atom slot (a forcefield type of
// the ligand set) and group the pair coefficients and the squared distances
// beyond which the pair's hinges are exactly zero.
struct Scene {
  const float4 *protein = nullptr;
  const PairCoef *coef = nullptr;   // [nslots][ngroups]
  // [nslots + 1][ngroups]: steric, charge, desolvation (-1: weight 0), their
  // largest; the last row the largest of every slot in w
  const float4 *reach2 = nullptr;
  int natpro = 0, ngroups = 0;
  int form = 1;                     // hinge form (plain_form())
  float lo[3] = {}, hi[3] = {};     // the protein's box, widened by the largest reach
};

// n poses of one ligand, rows pose_off .. pose_off + n - 1 of the pose
// arrays (or of the index into them); their energies go to the same rows.
struct Segment {
  int32_t lig;
  int64_t pose_off;
  int64_t n;
};

// Distances beyond which a pair's steric, charge and desolvation hinges are
// exactly zero in either hinge form: their zero crossings, widened far above
// the rounding of the distances compared with them; -1 for a hinge of weight
// 0.  False when the pair has no such distances (a radius sum that is not
// positive, or a coefficient that is not finite), so that no pair may be left
// out.
bool pair_reach(const PairCoef &c, float r[3]);

// The squared reaches of a coefficient table (Scene::reach2) and the largest
// reach; false when some pair has none.
bool reach_table(const std::vector<PairCoef> &coef, size_t ngroups, std::vector<float4> &reach2, float *largest);

// The box of the grouped protein's finite atoms widened by `reach`.
void protein_box(const std::vector<float> &xyzw, float reach, float lo[3], float hi[3]);

// The work of a pass: `items` items of `poses` poses in nsegs segments.
struct Work {
  size_t natpro = 0, ngroups = 0, nsegs = 0;
  double items = 0, poses = 0;
};

// Whether sorting pays, and whether the direct pass does, where the other
// choice is a tiled kernel with ppwi poses per work-item in register blocks of rb.
// pose_ps: the tiled kernel's cost of a pose besides its items' (kPlainPose,
// or the persistent kernel's), in ps of the whole device.
constexpr double kPlainPose = 8.0;
inline double persistent_pose(int rb) { return 40.0 + 160.0 / rb; }
bool worth_sorting(const Work &w, int ppwi, int rb, double pose_ps = kPlainPose);
// passes: launches the direct pass is split into; wait_us: what the tiled kernel costs more than its launch.
bool worth_direct(const Work &w, int ppwi, int rb, size_t passes = 1, double wait_us = 0.0);

// Device scratch of a pass; one stream at a time may use it.
struct Workspace {
  DeviceBuffer buf;
};

// The work of one pass, split into chunks of at most kChunkItems items.
class Plan {
 public:
  // atoms: every ligand's atoms (w bits: slot), ligand l's at lig_off[l] ..
  // lig_off[l + 1] - 1.  The tables are uploaded synchronously; no pass over
  // an earlier plan may be in flight.  A ligand too large for a chunk, or no
  // memory for the tables, leaves the plan empty().
  int build(const std::vector<float4> &atoms, const std::vector<int32_t> &lig_off, int nslots,
            const std::vector<Segment> &segs);
  // Grows w to what a pass needs.  Without the memory for it w is what it was
  // (or empty), and the status says so: ask fits() before every pass.
  int reserve(Workspace &w) const;
  bool fits(const Workspace &w) const { return w.buf.bytes >= layout()[6]; }
  // Queues the pass: energies[row] of every row of every segment.  index:
  // the pose row of row i of a segment is pose_off + index[pose_off + i].
  hipError_t launch(const Scene &sc, const Workspace &w, const float *poses, size_t stride, const uint32_t *index,
                    float *energies, hipStream_t s) const;
  bool worth(size_t natpro, size_t ngroups, int ppwi, double pose_ps) const {
    return !chunks_.empty() && worth_sorting(Work{natpro, ngroups, nsegs_, items_, poses_}, ppwi, ppwi, pose_ps);
  }
  bool empty() const { return chunks_.empty(); }
  void clear() {
    chunks_.clear();
    tables_.reset();
    atoms_.reset();
  }

 private:
  struct Chunk {
    int nblocks, ntasks, nslots_rows, ppt, rb, cell_bits;
    size_t blocks, tasks, refs, rows, slot_rows, slot_items, slot_units;  // offsets into tables_
    uint32_t nitems, npartial, nxform, nrows;
    int nunits;
  };
  // offsets of items, partial, xform, hist, base and bounds in the workspace, and its size
  std::array<size_t, 7> layout() const;
  std::vector<Chunk> chunks_;
  DeviceBuffer tables_, atoms_;
  int nslots_ = 0;
  size_t nsegs_ = 0;
  float radius_ = 0.f;  // of the ligand atoms about their frame's origin
  double items_ = 0, poses_ = 0;
};

// Single atoms at given points, sorted once and scored against any number of
// scenes with the same slots: out[i] is the plain kernel's energy of a
// one-atom ligand at point i, bit for bit.
class Points {
 public:
  // n points on the device, either packed (x, y, z, slot bits) or as
  // coordinates xyz[3 i ..] and slots[i]; slot_count[s] of them have slot s.
  // Queued on s; the inputs are read by the queued kernels only.
  int build(const float4 *packed, const float *xyz, const int32_t *slots, size_t n,
            const std::vector<size_t> &slot_count, hipStream_t s);
  hipError_t launch(const Scene &sc, float *out, hipStream_t s) const;

 private:
  DeviceBuffer buf_;
  const float4 *items_ = nullptr;
  const int32_t *slot_items_ = nullptr, *slot_units_ = nullptr;
  int nslots_ = 0, nunits_ = 0, rb_ = 1;
};

// The pass over every pair, for decks too small to sort (and those whose
// pairs have no reach): one wave per 64 poses and ligand atom or, while those
// are too few for the device, several that share the protein's groups; then the sums in
// the tiled kernels' order, so the energies are theirs bit for bit.
struct DirectArgs {
  const float4 *protein;
  const int32_t *group_begin;  // ngroups + 1
  const PairCoef *coef;        // [natlig][ngroups]
  const float4 *ligand;
  const float *poses;          // 6 rows of `stride` floats
  float *energies;             // nposes
  size_t stride, nposes;
  int natlig, ngroups, form;
  const int32_t *skip;         // device flag: nothing is scored when set (may be null)
  float *scratch;              // direct_bytes(nposes, natlig)
};
// Scratch of a direct pass over n poses.  Above kDirectBytes the tiled kernel
// scores as fast without it.
constexpr size_t kDirectBytes = size_t(64) << 20;
size_t direct_bytes(size_t n, size_t natlig);
hipError_t launch_direct(const DirectArgs &a, hipStream_t s);

// Everything one deck's passes need on the sorted path, from the host deck:
// scene, plan and workspace.  usable() is false where the path does not
// apply (see worth_sorting, pair_reach) or its memory cannot be had, worth()
// where a tiled kernel is the faster; the caller then scores with that.
class Deck {
 public:
  int prepare(const ProteinGroups &groups, const BudeFFParams *ff, const std::vector<BudeAtom> &atoms,
              const std::vector<int32_t> &lig_off, const std::vector<Segment> &segs);
  bool usable() const { return usable_; }
  bool worth(int ppwi, int rb, double pose_ps = kPlainPose) const {
    return usable_ && worth_sorting(shape_, ppwi, rb, pose_ps);
  }
  // Not usable() any more, and holding no memory.
  void release();
  hipError_t launch(const float4 *protein, const float *poses, size_t stride, const uint32_t *index, float *energies,
                    hipStream_t s) const;

 private:
  // prepare() up to *ok, whether there is a pass to run
  int plan(const ProteinGroups &groups, const BudeFFParams *ff, const std::vector<BudeAtom> &atoms,
           const std::vector<int32_t> &lig_off, const std::vector<Segment> &segs, bool *ok);
  bool usable_ = false;
  Work shape_;
  Scene scene_;
  Plan plan_;
  Workspace work_;
  DeviceBuffer coef_, reach2_;
};

}  // namespace items
}  // namespace bude
