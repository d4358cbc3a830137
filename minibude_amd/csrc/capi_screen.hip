// capi_screen.hip -- C ABI of the learned prescreen: an MLP pose-energy
// surrogate trained on the GPU (own BF16-MFMA forward/backward kernels,
// Adam) on energies the plain kernel computes, then used to screen a pose
// set: surrogate on every pose, exact plain-kernel rescoring of the lowest
// keep_fraction, plain kernel on everything when the surrogate's validation
// error is above the configured bound (fallback).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "bude_internal.h"
#include "fasten_batch.h"
#include "fasten_plain.h"
#include "hip_util.h"
#include "items.h"
#include "mlp.h"
#include "select.h"
#include "surrogate.h"

namespace {

using bude::DeviceBuffer;
using bude::mlp::bf16;
using bude::surrogate::Acts;
using bude::surrogate::Net;
using bude::surrogate::kK;
using bude::surrogate::kN;

double ms_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace

struct bude_screen {
  int device = 0;
  int cus = 0;
  size_t lds_per_cu = 0;
  BudeScreenConfig cfg{};
  // plain-kernel deck (labels, rescoring, fallback)
  size_t natlig = 0, ngroups = 0;
  DeviceBuffer protein, group_begin, coef, ligand;
  bude::ProteinGroups groups;
  std::vector<BudeAtom> atoms;
  std::vector<BudeFFParams> ff;
  // surrogate
  Net net;
  bool trained = false, fallback = false;
  float clip = 0.f, mu = 0.f, sigma = 1.f, tail = -3.0e38f, val_rmse = 0.f;
  // candidate poses
  size_t ncand = 0;
  DeviceBuffer cand, pred, sel_idx, sel_n, exact;
  // rescoring: rows through sel_idx, one ligand whose pose count and tiles
  // (first pose of 64) the device writes from the selection's size
  DeviceBuffer rs_tiles, rs_meta, rs_counter, rs_order, rs_ntiles;
  bude::sel::Plan plan;  // one segment: the loaded poses, k = ceil(keep_fraction * n)
  size_t plan_n = 0, plan_k = 0;
  // the sorted passes over the selection's first plan_k rows (the tiled
  // kernel scores rows past them: ties) and, in fallback, over every pose
  bude::items::Deck sel_deck, all_deck;
  DeviceBuffer rs_done;
  bool all_planned = false;
  size_t nsel = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev[5] = {};

  ~bude_screen() {
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }

  // The sorted passes' memory given back; the next run plans anew.
  void release_plans() {
    plan_n = 0;
    all_planned = false;
    sel_deck.release();
    all_deck.release();
  }

  bude::PlainArgs plain(const float *poses, size_t stride, size_t n, float *energies) const {
    bude::PlainArgs a{};
    a.protein = static_cast<const float4 *>(protein.ptr);
    a.group_begin = static_cast<const int32_t *>(group_begin.ptr);
    a.coef = static_cast<const bude::PairCoef *>(coef.ptr);
    a.ligand = static_cast<const float4 *>(ligand.ptr);
    a.poses = poses;
    a.energies = energies;
    a.stride = stride;
    a.nposes = n;
    a.natlig = int(natlig);
    a.ngroups = int(ngroups);
    a.ppwi = 1;
    a.form = bude::plain_form();
    return a;
  }
};

namespace {

// The sorted pass over rows [0, n) of a pose set (or of an index into one).
int plan_deck(const bude_screen *s, size_t n, bude::items::Deck &d) {
  return d.prepare(s->groups, s->ff.data(), s->atoms, {0, int32_t(s->natlig)},
                   {bude::items::Segment{0, 0, int64_t(n)}});
}

// Exact energies of n poses on the library's stream, through the planned
// pass where it applies.
hipError_t score_all(const bude_screen *s, const bude::items::Deck &d, const float *poses, size_t n, float *energies) {
  if (d.worth(1, 1))
    return d.launch(static_cast<const float4 *>(s->protein.ptr), poses, n, nullptr, energies, s->stream);
  return bude::launch_plain(s->plain(poses, n, n, energies), 256, s->stream);
}

int upload_poses(DeviceBuffer &d, const float *const poses[6], size_t n) {
  if (int st = d.alloc(6 * n * sizeof(float))) return st;
  for (int k = 0; k < 6; k++)
    if (int st = bude::hip_check(hipMemcpy(static_cast<float *>(d.ptr) + size_t(k) * n, poses[k], n * sizeof(float),
                                           hipMemcpyHostToDevice),
                                 "hipMemcpy poses"))
      return st;
  return BUDE_OK;
}

// Exact energies of the selected poses (rows sel_idx[0, nsel) of the
// candidates) into exact[0, nsel): the sorted pass over the plan_k rows that
// are always there, where it applies, and work-groups per 64 poses or the
// persistent kernel (bit-identical) over the rest.  The tables come from the selection's count
// on the device; the host does not wait for it.
int rescore(bude_screen *s) {
  const bool sorted = s->sel_deck.worth(1, 1);
  if (sorted)
    if (int st = bude::hip_check(s->sel_deck.launch(static_cast<const float4 *>(s->protein.ptr),
                                                    static_cast<const float *>(s->cand.ptr), s->ncand,
                                                    static_cast<const uint32_t *>(s->sel_idx.ptr),
                                                    static_cast<float *>(s->exact.ptr), s->stream),
                                 "sorted rescoring"))
      return st;
  if (int st = bude::hip_check(bude::build_rescore_tables(static_cast<const int32_t *>(s->rs_order.ptr), 1,
                                                          static_cast<const uint32_t *>(s->sel_n.ptr),
                                                          sorted ? static_cast<const uint32_t *>(s->rs_done.ptr)
                                                                 : nullptr,
                                                          static_cast<bude::LigandMeta *>(s->rs_meta.ptr),
                                                          static_cast<int2 *>(s->rs_tiles.ptr),
                                                          static_cast<int32_t *>(s->rs_ntiles.ptr), s->stream),
                               "rescoring tables"))
    return st;
  bude::BatchArgs a{};
  a.protein = static_cast<const float4 *>(s->protein.ptr);
  a.group_begin = static_cast<const int32_t *>(s->group_begin.ptr);
  a.coef = static_cast<const bude::PairCoef *>(s->coef.ptr);
  a.ligands = static_cast<const float4 *>(s->ligand.ptr);
  a.meta = static_cast<const bude::LigandMeta *>(s->rs_meta.ptr);
  a.tiles = static_cast<const int2 *>(s->rs_tiles.ptr);
  a.poses = static_cast<const float *>(s->cand.ptr);
  a.energies = static_cast<float *>(s->exact.ptr);
  a.stride = s->ncand;
  a.ngroups = int(s->ngroups);
  a.form = bude::plain_form();
  a.pose_index = static_cast<const uint32_t *>(s->sel_idx.ptr);
  a.ntiles_dev = static_cast<const int32_t *>(s->rs_ntiles.ptr);
  bude::TileWork work;  // what is expected: the tiles are counted on the device
  if (!sorted) work.add(s->natlig, s->plan_k);
  if (bude::worth_tiles(work, s->groups.xyzw.size() / 4, s->ngroups))
    return bude::hip_check(bude::launch_tiles(a, 2 * s->cus, s->stream), "rescore launch");
  a.counter = static_cast<unsigned int *>(s->rs_counter.ptr);
  const bude::PinnedGrid g = bude::pinned_grid(s->cus, s->lds_per_cu, 3);
  a.lds_bytes = g.lds_bytes;
  return bude::hip_check(bude::launch_batch_indexed(a, g.blocks, s->stream), "rescore launch");
}

// Surrogate predictions (normalised target units) for n poses whose 6 rows
// start at `poses` with row stride `stride`: the fused inference kernel on a
// persistent grid of 2 work-groups per CU.
int predict_all(bude_screen *s, const float *poses, size_t stride, size_t n, float *out) {
  if (int st = bude::surrogate::predict(s->net, poses, stride, n, out, 2 * s->cus, s->stream)) return st;
  return bude::hip_check(hipStreamSynchronize(s->stream), "hipStreamSynchronize");
}

}  // namespace

extern "C" int bude_mi355x_screen_create(int device, const BudeAtom *protein, size_t natpro, const BudeAtom *ligand,
                                         size_t natlig, const BudeFFParams *forcefield, size_t ntypes,
                                         const BudeScreenConfig *cfg, bude_screen **out) {
  if (!out || !cfg) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_create: NULL argument");
  *out = nullptr;
  if (int st = bude::check_deck(protein, natpro, ligand, natlig, forcefield, ntypes, "bude_mi355x_screen_create"))
    return st;
  if (cfg->batch < 32 || cfg->batch % 32 || cfg->batch > (1u << 20) || !(cfg->keep_fraction > 0.f) ||
      cfg->keep_fraction > 1.f || !(cfg->lr > 0.f) || !(cfg->clip_quantile > 0.f) || cfg->clip_quantile > 1.f ||
      cfg->tail_quantile < 0.f || cfg->tail_quantile > 1.f || !(cfg->tail_weight > 0.f) ||
      (cfg->features != 12 && cfg->features != uint32_t(bude::mlp::kFeat)))
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT,
                      "bude_mi355x_screen_create: batch must be a multiple of 32 in [32, 2^20], keep_fraction and "
                      "clip_quantile in (0, 1], tail_quantile in [0, 1], lr > 0, tail_weight > 0, features 12 or 21");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0 || device < 0 || device >= ndev)
    return bude::fail(BUDE_ERR_NO_DEVICE, "bude_mi355x_screen_create: no such HIP device");
  if (int st = bude::hip_check(hipSetDevice(device), "hipSetDevice")) return st;

  auto s = std::make_unique<bude_screen>();
  s->device = device;
  s->cfg = *cfg;
  hipDeviceProp_t props{};
  if (int st = bude::hip_check(hipGetDeviceProperties(&props, device), "hipGetDeviceProperties")) return st;
  s->cus = props.multiProcessorCount;
  s->lds_per_cu = props.maxSharedMemoryPerMultiProcessor;
  s->natlig = natlig;
  s->atoms.assign(ligand, ligand + natlig);
  s->ff.assign(forcefield, forcefield + ntypes);
  s->groups = bude::group_protein(protein, natpro);
  const bude::ProteinGroups &groups = s->groups;
  s->ngroups = groups.ngroups();
  const std::vector<bude::PairCoef> coef = bude::coef_table(ligand, natlig, groups, forcefield);
  std::vector<float> lig4(natlig * 4);
  for (size_t i = 0; i < natlig; i++) {
    lig4[4 * i + 0] = ligand[i].x;
    lig4[4 * i + 1] = ligand[i].y;
    lig4[4 * i + 2] = ligand[i].z;
  }
  int st = s->protein.upload(groups.xyzw.data(), groups.xyzw.size() * 4);
  if (!st) st = s->group_begin.upload(groups.begin.data(), groups.begin.size() * 4);
  if (!st) st = s->coef.upload(coef.data(), coef.size() * sizeof(bude::PairCoef));
  if (!st) st = s->ligand.upload(lig4.data(), lig4.size() * 4);
  if (!st) st = s->sel_n.alloc(256);
  if (!st) st = bude::hip_check(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking), "hipStreamCreate");
  for (auto &e : s->ev)
    if (!st) st = bude::hip_check(hipEventCreate(&e), "hipEventCreate");
  std::vector<std::vector<float>> w, b;
  // (with 12 inputs the first-layer rows of the rotation entries start at
  // zero and, their inputs being zero in training, stay there)
  bude::surrogate::init_weights(cfg->seed, int(cfg->features), w, b);
  if (!st) st = bude::surrogate::set_weights(s->net, w, b, s->stream);
  if (st) return st;
  *out = s.release();
  return bude::ok();
}

extern "C" int bude_mi355x_screen_train(bude_screen *s, const float *const poses[6], size_t n,
                                        BudeScreenTrainStats *stats, float *loss_curve, size_t loss_cap) {
  if (!s || !poses || !stats) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_train: NULL argument");
  const size_t B = s->cfg.batch;
  const size_t nval = std::max<size_t>(32, n / 16);
  if (n < 2 * B + nval || n > 0xffffffffu)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_train: need at least 2 batches + a validation "
                                                 "split (n/16) of poses");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  *stats = BudeScreenTrainStats{};
  hipStream_t st_ = s->stream;

  // 1. exact labels from the plain kernel
  s->release_plans();  // (training needs the memory more)
  DeviceBuffer tp, te;
  if (int st = upload_poses(tp, poses, n)) return st;
  if (int st = te.alloc(n * 4)) return st;
  auto t0 = std::chrono::steady_clock::now();
  {
    bude::items::Deck d;
    if (int st = plan_deck(s, n, d)) return st;
    if (int st = bude::hip_check(
            score_all(s, d, static_cast<const float *>(tp.ptr), n, static_cast<float *>(te.ptr)), "label launch"))
      return st;
    if (int st = bude::hip_check(hipStreamSynchronize(st_), "hipStreamSynchronize")) return st;
  }
  stats->label_ms = ms_since(t0);

  // 2. target transform from the training split: clip at a quantile (the
  //    screen ranks the low tail), standardise
  const size_t ntrain = n - nval;
  std::vector<float> e(n);
  if (int st = bude::hip_check(hipMemcpy(e.data(), te.ptr, n * 4, hipMemcpyDeviceToHost), "hipMemcpy")) return st;
  {
    std::vector<float> sorted(e.begin(), e.begin() + long(ntrain));
    const size_t q = std::min(ntrain - 1, size_t(double(s->cfg.clip_quantile) * double(ntrain)));
    std::nth_element(sorted.begin(), sorted.begin() + long(q), sorted.end());
    s->clip = sorted[q];
    if (s->cfg.tail_quantile > 0.f) {
      const size_t qt = std::min(ntrain - 1, size_t(double(s->cfg.tail_quantile) * double(ntrain)));
      std::nth_element(sorted.begin(), sorted.begin() + long(qt), sorted.end());
      s->tail = sorted[qt];
    }
    double sum = 0, sq = 0;
    for (size_t i = 0; i < ntrain; i++) {
      const double y = std::min(e[i], s->clip);
      sum += y;
      sq += y * y;
    }
    s->mu = float(sum / double(ntrain));
    s->sigma = float(std::sqrt(std::max(1e-12, sq / double(ntrain) - double(s->mu) * s->mu)));
  }

  // 3. Adam over shuffled mini-batches of the training split
  std::vector<uint32_t> perm(ntrain);
  std::iota(perm.begin(), perm.end(), 0u);
  bude::surrogate::TrainData td;
  td.poses = static_cast<const float *>(tp.ptr);
  td.stride = n;
  td.energy = static_cast<const float *>(te.ptr);
  td.norm = bude::mlp::TargetNorm{s->clip, s->mu, 1.0f / s->sigma, s->tail};
  td.nfeat = int(s->cfg.features);
  bude::surrogate::TrainParams tpar;
  tpar.batch = uint32_t(B);
  tpar.epochs = s->cfg.epochs;
  tpar.lr = s->cfg.lr;
  tpar.tail_weight = s->cfg.tail_weight;
  tpar.seed = s->cfg.seed;
  bude::surrogate::TrainReport rep;
  t0 = std::chrono::steady_clock::now();
  if (int st = bude::surrogate::train(s->net, td, std::move(perm), tpar, st_, loss_curve, loss_cap, &rep)) return st;
  stats->final_loss = rep.final_loss;
  stats->train_ms = ms_since(t0);
  stats->steps = rep.steps;

  // 4. validation RMSE (normalised units) on the held-out split
  DeviceBuffer vpred;
  if (int st = vpred.alloc(nval * 4)) return st;
  if (int st = predict_all(s, static_cast<const float *>(tp.ptr) + ntrain, n, nval, static_cast<float *>(vpred.ptr)))
    return st;
  {
    std::vector<float> vp(nval);
    if (int st = bude::hip_check(hipMemcpy(vp.data(), vpred.ptr, nval * 4, hipMemcpyDeviceToHost), "hipMemcpy"))
      return st;
    double se = 0;
    for (size_t i = 0; i < nval; i++) {
      const double y = (double(std::min(e[ntrain + i], s->clip)) - s->mu) / s->sigma;
      se += (vp[i] - y) * (vp[i] - y);
    }
    s->val_rmse = float(std::sqrt(se / double(nval)));
  }
  s->trained = true;
  s->fallback = !(s->val_rmse <= s->cfg.max_val_rmse);
  stats->val_rmse = s->val_rmse;
  stats->clip = s->clip;
  stats->mu = s->mu;
  stats->sigma = s->sigma;
  stats->fallback = s->fallback ? 1 : 0;
  return bude::ok();
}

extern "C" int bude_mi355x_screen_load(bude_screen *s, const float *const poses[6], size_t n) {
  if (!s || !poses || n == 0 || n > 0xffffffffu)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_load: bad arguments");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  s->ncand = n;
  s->nsel = 0;
  s->release_plans();
  int st = upload_poses(s->cand, poses, n);
  if (!st) st = s->pred.alloc(n * 4);
  if (!st) st = s->sel_idx.alloc(n * 4);
  if (!st) st = s->exact.alloc(n * 4);
  if (!st) st = s->rs_tiles.alloc((n + 63) / 64 * sizeof(int2));
  if (!st) st = s->rs_counter.alloc(sizeof(unsigned int));
  if (!st) st = s->rs_ntiles.alloc(sizeof(int32_t));
  if (!st) {  // the one ligand's row of the rescoring meta (its pose count comes from the selection)
    const bude::LigandMeta m{0, int32_t(s->natlig), 0, 0, 0, 0};
    st = s->rs_meta.assign(&m, sizeof(m));
  }
  if (!st) {
    const int32_t zero = 0;
    st = s->rs_order.assign(&zero, sizeof(zero));
  }
  return st;
}

extern "C" int bude_mi355x_screen_run(bude_screen *s, BudeScreenResult *res) {
  if (!s || !res) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_run: NULL argument");
  if (!s->trained || s->ncand == 0)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_run: train and load poses first");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  *res = BudeScreenResult{};
  const size_t n = s->ncand;
  const size_t k = std::max<size_t>(1, size_t(std::ceil(double(s->cfg.keep_fraction) * double(n))));
  hipStream_t st_ = s->stream;
  const auto t0 = std::chrono::steady_clock::now();
  if (s->plan_n != n || s->plan_k != k) {  // (uploads before any launch of this run)
    s->plan_n = 0;
    if (int st = s->plan.prepare({bude::sel::Segment{0, uint32_t(n), uint32_t(k)}})) return st;
    const uint32_t done = uint32_t(k);
    if (int st = s->rs_done.assign(&done, sizeof(done))) return st;
    if (int st = plan_deck(s, k, s->sel_deck)) return st;
    s->plan_n = n;
    s->plan_k = k;
  }
  if (s->fallback && !s->all_planned) {
    if (int st = plan_deck(s, n, s->all_deck)) return st;
    s->all_planned = true;
  }
  float ms01 = 0, ms12 = 0, ms23 = 0;
  if (s->fallback) {
    // plain kernel on every pose, then the same selection on exact energies
    if (int st = bude::hip_check(hipEventRecord(s->ev[0], st_), "hipEventRecord")) return st;
    if (int st = bude::hip_check(score_all(s, s->all_deck, static_cast<const float *>(s->cand.ptr), n,
                                           static_cast<float *>(s->pred.ptr)),
                                 "fallback launch"))
      return st;
    if (int st = bude::hip_check(hipEventRecord(s->ev[1], st_), "hipEventRecord")) return st;
  } else {
    if (int st = bude::hip_check(hipEventRecord(s->ev[0], st_), "hipEventRecord")) return st;
    if (int st = bude::surrogate::predict(s->net, static_cast<const float *>(s->cand.ptr), n, n,
                                          static_cast<float *>(s->pred.ptr), 2 * s->cus, st_))
      return st;
    if (int st = bude::hip_check(hipEventRecord(s->ev[1], st_), "hipEventRecord")) return st;
  }
  if (int st = bude::hip_check(bude::sel::select_lowest_segments(s->plan, static_cast<const float *>(s->pred.ptr),
                                                                 static_cast<uint32_t *>(s->sel_idx.ptr),
                                                                 static_cast<uint32_t *>(s->sel_n.ptr), st_),
                               "select"))
    return st;
  if (int st = bude::hip_check(hipEventRecord(s->ev[2], st_), "hipEventRecord")) return st;
  if (!s->fallback)  // (in fallback the exact energies are already in pred)
    if (int st = rescore(s)) return st;
  if (int st = bude::hip_check(hipEventRecord(s->ev[3], st_), "hipEventRecord")) return st;
  uint32_t nsel = 0;
  if (int st = bude::hip_check(hipMemcpyAsync(&nsel, s->sel_n.ptr, 4, hipMemcpyDeviceToHost, st_), "hipMemcpyAsync"))
    return st;
  if (int st = bude::hip_check(hipStreamSynchronize(st_), "hipStreamSynchronize")) return st;
  s->nsel = nsel;
  (void)hipEventElapsedTime(&ms01, s->ev[0], s->ev[1]);
  (void)hipEventElapsedTime(&ms12, s->ev[1], s->ev[2]);
  (void)hipEventElapsedTime(&ms23, s->ev[2], s->ev[3]);
  res->total_ms = ms_since(t0);
  res->score_ms = ms01;
  res->select_ms = ms12;
  res->rescore_ms = ms23;
  res->nposes = n;
  res->nselected = nsel;
  res->fallback = s->fallback ? 1 : 0;
  return bude::ok();
}

extern "C" int bude_mi355x_screen_set_keep(bude_screen *s, float keep_fraction) {
  if (!s || !(keep_fraction > 0.f) || keep_fraction > 1.f)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_set_keep: keep_fraction must be in (0, 1]");
  s->cfg.keep_fraction = keep_fraction;
  return bude::ok();
}

extern "C" int bude_mi355x_screen_selected(bude_screen *s, uint32_t *idx, float *energies, size_t cap, size_t *n) {
  if (!s || !n) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_selected: NULL argument");
  *n = s->nsel;
  if (!idx && !energies) return bude::ok();
  if (cap < s->nsel) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_selected: buffer too small");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  std::vector<uint32_t> id(s->nsel);
  if (int st = bude::hip_check(hipMemcpy(id.data(), s->sel_idx.ptr, s->nsel * 4, hipMemcpyDeviceToHost), "hipMemcpy"))
    return st;
  std::vector<float> ex(s->nsel);
  if (s->fallback) {
    std::vector<float> all(s->ncand);
    if (int st = bude::hip_check(hipMemcpy(all.data(), s->pred.ptr, s->ncand * 4, hipMemcpyDeviceToHost), "hipMemcpy"))
      return st;
    for (size_t j = 0; j < s->nsel; j++) ex[j] = all[id[j]];
  } else if (s->nsel) {
    if (int st = bude::hip_check(hipMemcpy(ex.data(), s->exact.ptr, s->nsel * 4, hipMemcpyDeviceToHost), "hipMemcpy"))
      return st;
  }
  // (selections are in pose order)
  if (idx) std::copy(id.begin(), id.end(), idx);
  if (energies) std::copy(ex.begin(), ex.end(), energies);
  return bude::ok();
}

extern "C" int bude_mi355x_screen_predict(bude_screen *s, float *pred) {
  if (!s || !pred || s->ncand == 0)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_predict: load poses first");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  DeviceBuffer out;
  if (int st = out.alloc(s->ncand * 4)) return st;
  if (int st = predict_all(s, static_cast<const float *>(s->cand.ptr), s->ncand, s->ncand,
                           static_cast<float *>(out.ptr)))
    return st;
  std::vector<float> p(s->ncand);
  if (int st = bude::hip_check(hipMemcpy(p.data(), out.ptr, s->ncand * 4, hipMemcpyDeviceToHost), "hipMemcpy"))
    return st;
  for (size_t i = 0; i < s->ncand; i++) pred[i] = p[i] * s->sigma + s->mu;  // back to energy units (clipped scale)
  return bude::ok();
}

extern "C" int bude_mi355x_screen_exhaustive(bude_screen *s, float *energies, double *ms) {
  if (!s || s->ncand == 0) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_screen_exhaustive: no poses");
  if (int st = bude::hip_check(hipSetDevice(s->device), "hipSetDevice")) return st;
  DeviceBuffer out;
  int ast = out.alloc(s->ncand * 4);
  if (ast == BUDE_ERR_OUT_OF_MEMORY) {
    s->release_plans();
    ast = out.alloc(s->ncand * 4);
  }
  if (ast) return ast;
  bude::items::Deck d;
  if (int st = plan_deck(s, s->ncand, d)) return st;
  if (int st = bude::hip_check(hipEventRecord(s->ev[0], s->stream), "hipEventRecord")) return st;
  if (int st = bude::hip_check(
          score_all(s, d, static_cast<const float *>(s->cand.ptr), s->ncand, static_cast<float *>(out.ptr)),
          "exhaustive launch"))
    return st;
  if (int st = bude::hip_check(hipEventRecord(s->ev[1], s->stream), "hipEventRecord")) return st;
  if (int st = bude::hip_check(hipStreamSynchronize(s->stream), "hipStreamSynchronize")) return st;
  float t = 0.f;
  (void)hipEventElapsedTime(&t, s->ev[0], s->ev[1]);
  if (ms) *ms = t;
  if (energies)
    return bude::hip_check(hipMemcpy(energies, out.ptr, s->ncand * 4, hipMemcpyDeviceToHost), "hipMemcpy");
  return bude::ok();
}

extern "C" int bude_mi355x_screen_destroy(bude_screen *s) {
  if (!s) return bude::ok();
  (void)hipSetDevice(s->device);
  delete s;
  return bude::ok();
}

namespace {

// The device memory of a call, handed out in aligned pieces: one allocation,
// as an allocation and its release cost the host some 10 us each (the calls
// below took 40 and 59).
class Arena {
 public:
  template <class T> size_t add(size_t n) {
    const size_t at = bytes_;
    bytes_ += (n * sizeof(T) + 255) & ~size_t(255);
    return at;
  }
  int alloc() { return buf_.alloc(bytes_); }
  template <class T> T *at(size_t offset) const { return reinterpret_cast<T *>(static_cast<char *>(buf_.ptr) + offset); }

 private:
  size_t bytes_ = 0;
  DeviceBuffer buf_;
};

// A network handed in whole: its FP32 arrays and the copies the kernels read.
struct Handed {
  size_t w[4], b[4], wt[3], wx[3], w3;
  explicit Handed(Arena &m, bool training) {
    using namespace bude::mlp;
    for (int l = 0; l < 4; l++) {
      w[l] = m.add<float>(size_t(kRealK[l]) * kRealN[l]);
      b[l] = m.add<float>(size_t(kRealN[l]));
    }
    for (int l = 0; l < 3; l++) {
      wt[l] = m.add<bf16>(size_t(kK[l]) * kN[l]);
      wx[l] = training && l > 0 ? m.add<bf16>(size_t(kK[l]) * kN[l]) : 0;
    }
    w3 = m.add<bf16>(size_t(kK[3]) * kN[3]);
  }
  int upload(const Arena &m, const float *const weights[4], const float *const biases[4], hipStream_t s) const {
    using namespace bude::mlp;
    for (int l = 0; l < 4; l++) {
      if (int st = bude::hip_check(hipMemcpyAsync(m.at<float>(w[l]), weights[l],
                                                  size_t(kRealK[l]) * kRealN[l] * sizeof(float),
                                                  hipMemcpyHostToDevice, s),
                                   "hipMemcpyAsync weights"))
        return st;
      if (int st = bude::hip_check(hipMemcpyAsync(m.at<float>(b[l]), biases[l], size_t(kRealN[l]) * sizeof(float),
                                                  hipMemcpyHostToDevice, s),
                                   "hipMemcpyAsync biases"))
        return st;
    }
    return BUDE_OK;
  }
  bude::mlp::StageArgs stage_args(const Arena &m, bool training) const {
    bude::mlp::StageArgs a{};
    for (int l = 0; l < 4; l++) a.w[l] = m.at<float>(w[l]);
    for (int l = 0; l < 3; l++) {
      a.wt[l] = m.at<bf16>(wt[l]);
      a.wx[l] = training && l > 0 ? m.at<bf16>(wx[l]) : nullptr;
    }
    a.w3 = m.at<bf16>(w3);
    return a;
  }
};

int check_device(int device, const char *who) {
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0 || device < 0 || device >= ndev)
    return bude::fail(BUDE_ERR_NO_DEVICE, std::string(who) + ": no such HIP device");
  return bude::hip_check(hipSetDevice(device), "hipSetDevice");
}

// Waits for the work of a call before its memory goes, however the call ends.
struct Drain {
  hipStream_t s;
  ~Drain() { (void)hipStreamSynchronize(s); }
};

}  // namespace

// 8,192 rows: 1,280 us with a buffer, a clear and a copy for each array (59, 25
// and 20 of them), 466 us; the kernels take 42.
extern "C" int bude_mi355x_mlp_forward_backward(int device, size_t batch, const float *features, const float *target,
                                                const float *const weights[4], const float *const biases[4],
                                                float *pred, float *loss, float *const grad_w[4],
                                                float *const grad_b[4]) {
  using namespace bude::mlp;
  if (!features || !target || !weights || !biases || !pred || !loss || !grad_w || !grad_b || batch == 0 ||
      batch % 32 || batch > (1u << 16))
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT,
                      "bude_mi355x_mlp_forward_backward: bad arguments (batch a multiple of 32, <= 65536)");
  if (int st = check_device(device, "bude_mi355x_mlp_forward_backward")) return st;
  const hipStream_t s = nullptr;
  const size_t ld = t_ld(batch);
  const int splits = dw_splits(batch);
  Arena m;
  const Handed net(m, true);
  const size_t feat = m.add<float>(batch * kFeat), tgt = m.add<float>(batch);
  const size_t feat16 = m.add<bf16>(batch * kIn), feat_t = m.add<bf16>(ld * kIn), dz3_t = m.add<bf16>(ld * kOut);
  size_t a_t[3], dz_t[3], work[4], part[4];
  for (int l = 0; l < 3; l++) {
    a_t[l] = m.add<bf16>(ld * kHidden);
    dz_t[l] = m.add<bf16>(ld * kHidden);
  }
  for (int l = 0; l < 4; l++) {
    work[l] = m.add<float>(size_t(splits) * kK[l] * kN[l]);
    part[l] = m.add<float>(size_t(splits) * kN[l]);
  }
  // what comes back, in one piece: the loss sum, the gradients, the predictions
  const size_t loss_floats = sizeof(unsigned long long) / sizeof(float);
  const size_t nout = loss_floats + kGradCount + batch, out = m.add<float>(nout);
  if (int st = m.alloc()) return st;
  const Drain drain{s};
  if (int st = net.upload(m, weights, biases, s)) return st;
  if (int st = bude::hip_check(hipMemcpyAsync(m.at<float>(feat), features, batch * kFeat * sizeof(float),
                                              hipMemcpyHostToDevice, s),
                               "hipMemcpyAsync features"))
    return st;
  if (int st = bude::hip_check(hipMemcpyAsync(m.at<float>(tgt), target, batch * sizeof(float), hipMemcpyHostToDevice,
                                              s),
                               "hipMemcpyAsync targets"))
    return st;
  float *dout = m.at<float>(out);
  StageArgs sa = net.stage_args(m, true);
  sa.feat = m.at<float>(feat);
  sa.rows = batch;
  sa.ld_t = ld;
  sa.feat16 = m.at<bf16>(feat16);
  sa.feat_t = m.at<bf16>(feat_t);
  sa.dz3_t = m.at<bf16>(dz3_t);
  sa.loss = reinterpret_cast<unsigned long long *>(dout);
  if (int st = bude::hip_check(stage(sa, s), "mlp inputs")) return st;
  RowsArgs in{};
  in.feat = sa.feat16;
  in.n = batch;
  in.ld_t = ld;
  in.energy = m.at<float>(tgt);
  in.norm = TargetNorm{3.0e38f, 0.f, 1.f, -3.0e38f};
  in.tail_weight = 1.f;
  in.pred = dout + loss_floats + kGradCount;
  in.loss = sa.loss;
  in.feat_t = sa.feat_t;
  in.dz3_t = sa.dz3_t;
  for (int l = 0; l < 3; l++) {
    in.wt[l] = sa.wt[l];
    in.a_t[l] = m.at<bf16>(a_t[l]);
    in.dz_t[l] = m.at<bf16>(dz_t[l]);
  }
  for (int l = 0; l < 4; l++) {
    in.w[l] = l == 3 ? sa.w3 : sa.wx[l];  // (w[0] unused)
    in.bias[l] = m.at<float>(net.b[l]);
  }
  if (int st = bude::hip_check(rows(in, s), "mlp rows")) return st;
  DwArgs dw{};
  dw.count = 4;
  dw.k = batch;
  dw.ld = ld;
  dw.splits = splits;
  for (int l = 0; l < 4; l++)
    dw.d[l] = DwProduct{l == 0 ? in.feat_t : in.a_t[l - 1], l == 3 ? in.dz3_t : in.dz_t[l], kK[l], kN[l],
                        m.at<float>(work[l]), m.at<float>(part[l])};
  if (int st = bude::hip_check(weight_grads(dw, s), "mlp weight gradients")) return st;
  if (int st = bude::hip_check(grads_out(dw, dout + loss_floats, s), "mlp gradients")) return st;
  const std::unique_ptr<float[]> host(new (std::nothrow) float[nout]);
  if (!host) return bude::fail(BUDE_ERR_OUT_OF_MEMORY, "bude_mi355x_mlp_forward_backward: no host memory");
  if (int st = bude::hip_check(hipMemcpyAsync(host.get(), dout, nout * sizeof(float), hipMemcpyDeviceToHost, s),
                               "hipMemcpyAsync"))
    return st;
  if (int st = bude::hip_check(hipStreamSynchronize(s), "hipStreamSynchronize")) return st;
  unsigned long long lsum = 0;
  std::memcpy(&lsum, host.get(), sizeof lsum);
  *loss = float(double(lsum) / kLossScale / double(batch));
  const float *p = host.get() + loss_floats;
  for (int l = 0; l < 4; l++) {
    const size_t n = size_t(kRealK[l]) * kRealN[l];
    std::copy(p, p + n, grad_w[l]);
    p += n;
  }
  for (int l = 0; l < 4; l++) {
    std::copy(p, p + kRealN[l], grad_b[l]);
    p += kRealN[l];
  }
  std::copy(p, p + batch, pred);
  return bude::ok();
}

// Poses from which the next poses are copied in and the last predictions out
// while a piece of them is scored: 2^20 poses 1,650 us in one piece, 1,340 in
// four, 1,380 in two, 1,530 in eight.
constexpr size_t kPredictPiece = size_t(1) << 18;

extern "C" int bude_mi355x_mlp_predict(int device, const float *const poses[6], size_t n,
                                       const float *const weights[4], const float *const biases[4], float *pred) {
  if (!poses || !weights || !biases || !pred || n == 0 || n > 0xffffffffu)
    return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_mlp_predict: bad arguments");
  if (int st = check_device(device, "bude_mi355x_mlp_predict")) return st;
  int cus = 0;
  if (int st = bude::hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device),
                               "hipDeviceGetAttribute"))
    return st;
  Arena m;
  const Handed net(m, false);
  const size_t dposes = m.add<float>(6 * n), dout = m.add<float>(n);
  if (int st = m.alloc()) return st;
  // copies in on the default stream; kernels and copies out behind them, on a
  // stream of their own where there are several pieces
  struct Side {
    hipStream_t s = nullptr;
    hipEvent_t ready = nullptr;
    ~Side() {
      (void)hipStreamSynchronize(nullptr);
      if (s) {
        (void)hipStreamSynchronize(s);
        (void)hipStreamDestroy(s);
      }
      if (ready) (void)hipEventDestroy(ready);
    }
  } side;
  if (n > kPredictPiece) {
    if (int st = bude::hip_check(hipStreamCreateWithFlags(&side.s, hipStreamNonBlocking), "hipStreamCreate")) return st;
    if (int st = bude::hip_check(hipEventCreateWithFlags(&side.ready, hipEventDisableTiming), "hipEventCreate"))
      return st;
  }
  if (int st = net.upload(m, weights, biases, nullptr)) return st;
  const bude::mlp::StageArgs sa = net.stage_args(m, false);
  if (int st = bude::hip_check(bude::mlp::stage(sa, nullptr), "mlp inputs")) return st;
  const bf16 *wt[4] = {sa.wt[0], sa.wt[1], sa.wt[2], nullptr};
  const float *bias[4] = {m.at<float>(net.b[0]), m.at<float>(net.b[1]), m.at<float>(net.b[2]), m.at<float>(net.b[3])};
  float *dp = m.at<float>(dposes), *out = m.at<float>(dout);
  auto fetch = [&](size_t first) {
    return bude::hip_check(hipMemcpyAsync(pred + first, out + first, std::min(kPredictPiece, n - first) * sizeof(float),
                                          hipMemcpyDeviceToHost, side.s),
                           "hipMemcpyAsync predictions");
  };
  size_t last = 0;
  for (size_t first = 0; first < n; first += kPredictPiece) {
    const size_t k = std::min(kPredictPiece, n - first);
    for (int r = 0; r < 6; r++)
      if (int st = bude::hip_check(hipMemcpyAsync(dp + size_t(r) * n + first, poses[r] + first, k * sizeof(float),
                                                  hipMemcpyHostToDevice, nullptr),
                                   "hipMemcpyAsync poses"))
        return st;
    if (side.s) {
      if (int st = bude::hip_check(hipEventRecord(side.ready, nullptr), "hipEventRecord")) return st;
      if (first)
        if (int st = fetch(last)) return st;
      if (int st = bude::hip_check(hipStreamWaitEvent(side.s, side.ready, 0), "hipStreamWaitEvent")) return st;
    }
    if (int st = bude::hip_check(bude::mlp::infer(dp + first, n, k, wt, sa.w3, bias, out + first, 2 * cus, side.s),
                                 "mlp infer"))
      return st;
    last = first;
  }
  if (int st = fetch(last)) return st;
  return bude::hip_check(hipStreamSynchronize(side.s), "hipStreamSynchronize");
}
