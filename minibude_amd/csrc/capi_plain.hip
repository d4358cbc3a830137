// capi_plain.hip -- C ABI of the plain fasten_main (devices, tunables,
// context lifecycle, timed launches).  Host code; the kernels live in
// fasten_plain.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <string>

#include "bude_internal.h"
#include "fasten_plain.h"
#include "hip_util.h"
#include "items.h"

namespace {

constexpr size_t kPpwi[] = {1, 2, 4, 8, 16, 32, 64, 128};  // src/main.cpp:48 DEFAULT_PPWI

bool ppwi_supported(size_t p) { return std::find(std::begin(kPpwi), std::end(kPpwi), p) != std::end(kPpwi); }
bool wgsize_supported(size_t w) { return w == 64 || w == 128 || w == 256 || w == 512 || w == 1024; }

constexpr size_t kHostResult = size_t(1) << 15;

double ms_since(std::chrono::steady_clock::time_point t0) {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace

struct bude_ctx {
  int device = 0;
  size_t natpro = 0, natlig = 0, ntypes = 0, nposes = 0, ngroups = 0;
  bude::DeviceBuffer protein, group_begin, coef, ligand, poses, energies;
  bude::items::Deck sorted;
  // scratch of the direct pass (null: not used): behind the energies, or by itself
  float *direct = nullptr;
  bude::DeviceBuffer direct_buf;
  // where the last pass of a call leaves its energies for the host to read
  // (not allocated: they are copied out)
  bude::PinnedBuffer result;
  bool in_result = false;   // the latest pass's energies are there, not in `energies`
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double context_ms = 0.0;

  bude::items::Work work() const {
    return {natpro, ngroups, 1, double(natlig) * double(nposes), double(nposes)};
  }

  ~bude_ctx() {
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

extern "C" int bude_mi355x_device_count(int *count) {
  if (!count) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_device_count: count is NULL");
  *count = 0;
  int n = 0;
  const hipError_t e = hipGetDeviceCount(&n);
  if (e == hipErrorNoDevice || (e == hipSuccess && n == 0))
    return bude::fail(BUDE_ERR_NO_DEVICE, "bude_mi355x_device_count: no HIP device visible");
  if (e != hipSuccess) return bude::hip_fail(e, "hipGetDeviceCount");
  *count = n;
  return bude::ok();
}

extern "C" int bude_mi355x_device_name(int device, char *buf, size_t len) {
  if (!buf || len == 0) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_device_name: empty buffer");
  hipDeviceProp_t props{};
  if (int st = bude::hip_check(hipGetDeviceProperties(&props, device), "hipGetDeviceProperties")) return st;
  // some runtimes leave the marketing name empty; fall back to the ISA name
  const std::string name = props.name[0] ? std::string(props.name) : std::string("AMD GPU ") + props.gcnArchName;
  const std::string s = name + " (" + std::to_string(props.totalGlobalMem / 1024 / 1024) + "MB;" +
                        props.gcnArchName + ";" + std::to_string(props.multiProcessorCount) + "CU)";
  std::strncpy(buf, s.c_str(), len - 1);
  buf[len - 1] = '\0';
  return bude::ok();
}

extern "C" int bude_mi355x_ppwi_list(size_t *out, size_t cap, size_t *count) {
  if (!count) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_ppwi_list: count is NULL");
  const size_t n = sizeof(kPpwi) / sizeof(kPpwi[0]);
  for (size_t i = 0; i < n && i < cap && out; i++) out[i] = kPpwi[i];
  *count = n;
  return bude::ok();
}

extern "C" int bude_mi355x_compatible(int device, size_t ppwi, size_t wgsize, int *ok) {
  if (!ok) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_compatible: ok is NULL");
  *ok = 0;
  if (!ppwi_supported(ppwi))
    return bude::fail(BUDE_ERR_UNSUPPORTED, "ppwi " + std::to_string(ppwi) + " is not one of 1,2,4,8,16,32,64,128");
  if (!wgsize_supported(wgsize))
    return bude::fail(BUDE_ERR_UNSUPPORTED,
                      "wgsize " + std::to_string(wgsize) + " is not one of 64,128,256,512,1024 (whole wavefronts)");
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n)
    return bude::fail(BUDE_ERR_NO_DEVICE, "device " + std::to_string(device) + " is not a visible HIP device");
  hipDeviceProp_t props{};
  if (int st = bude::hip_check(hipGetDeviceProperties(&props, device), "hipGetDeviceProperties")) return st;
  if (std::strncmp(props.gcnArchName, "gfx950", 6) != 0)
    return bude::fail(BUDE_ERR_UNSUPPORTED, std::string("device is ") + props.gcnArchName +
                                                ", the kernels are built for gfx950 only");
  *ok = 1;
  return bude::ok();
}

extern "C" int bude_mi355x_create(int device, const BudeAtom *protein, size_t natpro, const BudeAtom *ligand,
                                  size_t natlig, const BudeFFParams *forcefield, size_t ntypes,
                                  const float *const poses[6], size_t nposes, bude_ctx **out) {
  if (!out) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_create: out is NULL");
  *out = nullptr;
  if (int st = bude::check_deck(protein, natpro, ligand, natlig, forcefield, ntypes, "bude_mi355x_create")) return st;
  if (!poses || nposes == 0) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_create: no poses");
  for (int k = 0; k < 6; k++)
    if (!poses[k]) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_create: pose row is NULL");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return bude::fail(BUDE_ERR_NO_DEVICE, "bude_mi355x_create: no HIP device visible");
  if (device < 0 || device >= ndev)
    return bude::fail(BUDE_ERR_NO_DEVICE, "bude_mi355x_create: device " + std::to_string(device) + " out of range");

  const auto t0 = std::chrono::steady_clock::now();
  if (int st = bude::hip_check(hipSetDevice(device), "hipSetDevice")) return st;

  const bude::ProteinGroups groups = bude::group_protein(protein, natpro);
  const std::vector<bude::PairCoef> coef = bude::coef_table(ligand, natlig, groups, forcefield);
  std::vector<float> lig4(natlig * 4);
  for (size_t i = 0; i < natlig; i++) {
    lig4[4 * i + 0] = ligand[i].x;
    lig4[4 * i + 1] = ligand[i].y;
    lig4[4 * i + 2] = ligand[i].z;
    lig4[4 * i + 3] = 0.f;
  }

  auto *c = new bude_ctx();
  c->device = device;
  c->natpro = natpro;
  c->natlig = natlig;
  c->ntypes = ntypes;
  c->nposes = nposes;
  c->ngroups = groups.ngroups();
  int st = BUDE_OK;
  if (!st) st = c->protein.upload(groups.xyzw.data(), groups.xyzw.size() * sizeof(float));
  if (!st) st = c->group_begin.upload(groups.begin.data(), groups.begin.size() * sizeof(int32_t));
  if (!st) st = c->coef.upload(coef.data(), coef.size() * sizeof(bude::PairCoef));
  if (!st) st = c->ligand.upload(lig4.data(), lig4.size() * sizeof(float));
  if (!st) st = c->poses.alloc(6 * nposes * sizeof(float));
  for (int k = 0; k < 6 && !st; k++)
    st = bude::hip_check(hipMemcpy(static_cast<float *>(c->poses.ptr) + k * nposes, poses[k], nposes * sizeof(float),
                                   hipMemcpyHostToDevice),
                         "hipMemcpy poses");
  // A deck of a size that is not sorted has the direct pass's sums behind its
  // energies, where there is memory for both: a call's first pass over an
  // allocation of their own takes 5 us longer (64 poses 50 us, 45).
  const bude::items::Work work = c->work();
  const size_t direct = bude::items::direct_bytes(nposes, natlig), padded = (nposes + 63) / 64 * 64;
  const bool behind = direct <= bude::items::kDirectBytes && !bude::items::worth_sorting(work, 1, 1) &&
                      !bude::items::worth_sorting(work, 8, 8);
  if (!st) {
    st = c->energies.alloc(padded * sizeof(float) + (behind ? direct : 0));
    if (!st && behind) c->direct = static_cast<float *>(c->energies.ptr) + padded;
    if (st == BUDE_ERR_OUT_OF_MEMORY && behind) st = c->energies.alloc(nposes * sizeof(float));
  }
  if (!st) st = bude::hip_check(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "hipStreamCreate");
  if (!st) st = bude::hip_check(hipEventCreate(&c->ev0), "hipEventCreate");
  if (!st) st = bude::hip_check(hipEventCreate(&c->ev1), "hipEventCreate");
  // what a pass can do without comes last: the sorted pass's scratch, then the direct pass's
  if (!st)
    st = c->sorted.prepare(groups, forcefield, std::vector<BudeAtom>(ligand, ligand + natlig), {0, int32_t(natlig)},
                           {bude::items::Segment{0, 0, int64_t(nposes)}});
  if (!st && !c->sorted.usable() && !behind && direct <= bude::items::kDirectBytes) {
    st = c->direct_buf.alloc(direct);
    if (st == BUDE_ERR_OUT_OF_MEMORY) st = BUDE_OK;  // (the tiled kernel, then)
    c->direct = static_cast<float *>(c->direct_buf.ptr);
  }
  // A copy of few energies costs 12 us and more a call whatever their number;
  // the last pass stores them over the bus instead (a call of 64 poses 39 and
  // 27 us, 4,097 61 and 48, 16,384 97 and 91).  With more of them the memory
  // for it, pinned, costs more than calls gain soon (65,536: 150 and 140 us a
  // call, but 300 us here).  Only a pass that writes an energy once goes there.
  if (!st && nposes <= kHostResult && (c->sorted.usable() || c->direct)) {
    st = c->result.alloc(nposes * sizeof(float));
    if (st == BUDE_ERR_OUT_OF_MEMORY) st = BUDE_OK;  // (copied out, then)
  }
  if (!st) st = bude::hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
  if (st) {
    delete c;
    return st;
  }
  c->context_ms = ms_since(t0);
  *out = c;
  return bude::ok();
}

extern "C" int bude_mi355x_fasten(bude_ctx *ctx, size_t ppwi, size_t wgsize, size_t warmup, size_t iterations,
                                  float *energies_out, double *host_ms, double *device_ms) {
  if (!ctx) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_fasten: ctx is NULL");
  if (!ppwi_supported(ppwi))
    return bude::fail(BUDE_ERR_UNSUPPORTED, "ppwi " + std::to_string(ppwi) + " is not one of 1,2,4,8,16,32,64,128");
  if (!wgsize_supported(wgsize))
    return bude::fail(BUDE_ERR_UNSUPPORTED,
                      "wgsize " + std::to_string(wgsize) + " is not one of 64,128,256,512,1024 (whole wavefronts)");
  const size_t blocks = ((ctx->nposes + ppwi - 1) / ppwi + wgsize - 1) / wgsize;
  if (blocks > 0x7fffffffu) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_fasten: grid too large");
  if (int st = bude::hip_check(hipSetDevice(ctx->device), "hipSetDevice")) return st;

  bude::PlainArgs a{};
  a.protein = static_cast<const float4 *>(ctx->protein.ptr);
  a.group_begin = static_cast<const int32_t *>(ctx->group_begin.ptr);
  a.coef = static_cast<const bude::PairCoef *>(ctx->coef.ptr);
  a.ligand = static_cast<const float4 *>(ctx->ligand.ptr);
  a.poses = static_cast<const float *>(ctx->poses.ptr);
  a.energies = static_cast<float *>(ctx->energies.ptr);
  a.stride = ctx->nposes;
  a.nposes = ctx->nposes;
  a.natlig = int(ctx->natlig);
  a.ngroups = int(ctx->ngroups);
  a.ppwi = int(ppwi);
  a.form = bude::plain_form();
  bude::items::DirectArgs direct{a.protein, a.group_begin, a.coef,   a.ligand, a.poses, a.energies, a.stride,
                                 a.nposes,  a.natlig,      a.ngroups, a.form,   nullptr,
                                 ctx->direct};
  const size_t passes = warmup + iterations;
  // Few energies: the tiled kernel never pays, as they would be copied out.
  const bool few = ctx->nposes <= kHostResult;
  const int rb = bude::plain_register_block(int(ppwi), int(wgsize), ctx->nposes);
  const bool sorted = few ? ctx->sorted.usable() : ctx->sorted.worth(int(ppwi), rb);
  const bool use_direct = !sorted && ctx->direct && (few || bude::items::worth_direct(ctx->work(), int(ppwi), rb));

  for (size_t i = 0; i < passes; i++) {
    const bool to_host = energies_out && ctx->result.ptr && (sorted || use_direct) && i + 1 == passes;
    if (to_host) direct.energies = a.energies = static_cast<float *>(ctx->result.ptr);
    const auto t0 = std::chrono::steady_clock::now();
    if (int st = bude::hip_check(hipEventRecord(ctx->ev0, ctx->stream), "hipEventRecord")) return st;
    const hipError_t le =
        sorted       ? ctx->sorted.launch(a.protein, a.poses, a.stride, nullptr, a.energies, ctx->stream)
        : use_direct ? bude::items::launch_direct(direct, ctx->stream)
                     : bude::launch_plain(a, int(wgsize), ctx->stream);
    if (int st = bude::hip_check(le, "fasten_plain launch")) return st;
    if (int st = bude::hip_check(hipEventRecord(ctx->ev1, ctx->stream), "hipEventRecord")) return st;
    if (int st = bude::hip_check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize")) return st;
    ctx->in_result = to_host;
    if (host_ms) host_ms[i] = ms_since(t0);
    if (device_ms) {
      float ms = 0.f;
      if (int st = bude::hip_check(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1), "hipEventElapsedTime")) return st;
      device_ms[i] = ms;
    }
  }
  if (energies_out && ctx->in_result) {
    std::memcpy(energies_out, ctx->result.ptr, ctx->nposes * sizeof(float));
    return bude::ok();
  }
  if (energies_out)
    return bude::hip_check(
        hipMemcpy(energies_out, ctx->energies.ptr, ctx->nposes * sizeof(float), hipMemcpyDeviceToHost),
        "hipMemcpy energies");
  return bude::ok();
}

extern "C" int bude_mi355x_context_ms(const bude_ctx *ctx, double *ms) {
  if (!ctx || !ms) return bude::fail(BUDE_ERR_INVALID_ARGUMENT, "bude_mi355x_context_ms: NULL argument");
  *ms = ctx->context_ms;
  return bude::ok();
}

extern "C" int bude_mi355x_destroy(bude_ctx *ctx) {
  if (!ctx) return bude::ok();
  (void)hipSetDevice(ctx->device);
  delete ctx;
  return bude::ok();
}
