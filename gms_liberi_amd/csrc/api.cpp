// C ABI of the MI355X Fock build: handle lifecycle, setup, build.
//
// Host side of the drop-in for src/interface/liberi_interface.F90 (handle
// API), src/liberi_shell_pair.F90 (setup) and src/liberi_driver.F90
// (compute_integrals) of gms_libERI.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/liberi_hip.h"
#include "liberi_internal.hpp"

namespace liberi {

const ClassDef kClasses[kNumClasses] = {
    {"int0000", P_SS, P_SS, CMP_GE, PS_SELF},     {"int0001", P_SS, P_SP, CMP_GT, PS_CROSS},
    {"int0011", P_SS, P_PP, CMP_GT, PS_CROSS},    {"int0111", P_SP, P_PP, CMP_GT, PS_CROSS},
    {"int0101", P_SP, P_SP, CMP_GE, PS_SELF},     {"int1111", P_PP, P_PP, CMP_GE, PS_SELF},
    {"int0002", P_SS, P_SD, CMP_GT, PS_CROSS},    {"int0012", P_SS, P_PD, CMP_GT, PS_CROSS},
    {"int0102", P_SP, P_SD, CMP_GT, PS_CROSS},    {"int0112", P_SP, P_PD, CMP_GT, PS_CROSS},
    {"int0022", P_SS, P_DD, CMP_GT, PS_CROSS},    {"int0122", P_SP, P_DD, CMP_GT, PS_CROSS},
    {"int1102", P_PP, P_SD, CMP_GT, PS_CROSS},    {"int0202", P_SD, P_SD, CMP_GT, PS_SELF},
    {"int2211", P_DD, P_PP, CMP_GT, PS_SELF},     {"int2121", P_PD, P_PD, CMP_GT, PS_SELF},
    {"int2120", P_PD, P_SD, CMP_GT, PS_SELF},     {"int2111", P_PD, P_PP, CMP_GT, PS_SELF},
    {"int2220", P_DD, P_SD, CMP_GT, PS_SELF},     {"int2221", P_DD, P_PD, CMP_GT, PS_SELF},
    {"int2222gen", P_DD, P_DD, CMP_NONE, PS_SELF}, {"int3333", P_FF, P_FF, CMP_NONE, PS_SELF},
    {"int0030", P_SS, P_SF, CMP_GT, PS_SELF},     {"int0031", P_SS, P_PF, CMP_GT, PS_SELF},
    {"int0032", P_SS, P_DF, CMP_GT, PS_SELF},     {"int1030", P_SP, P_SF, CMP_GT, PS_SELF},
    {"int3330", P_FF, P_SF, CMP_GT, PS_SELF},     {"int3011", P_SF, P_PP, CMP_GT, PS_SELF},
    {"int3020", P_SF, P_SD, CMP_GT, PS_SELF},     {"int2130", P_PD, P_SF, CMP_GT, PS_SELF},
    {"int2230", P_DD, P_SF, CMP_GT, PS_SELF},     {"int3030", P_SF, P_SF, CMP_GT, PS_SELF},
    {"int3110", P_PF, P_SP, CMP_GT, PS_SELF},     {"int3111", P_PF, P_PP, CMP_GT, PS_SELF},
    {"int3120", P_PF, P_SD, CMP_GT, PS_SELF},     {"int3121", P_PF, P_PD, CMP_GT, PS_SELF},
    {"int2231", P_DD, P_PF, CMP_GT, PS_SELF},     {"int3130", P_PF, P_SF, CMP_GT, PS_SELF},
    {"int3131", P_PF, P_PF, CMP_GT, PS_SELF},     {"int3210", P_DF, P_SP, CMP_GT, PS_SELF},
    {"int3331", P_FF, P_PF, CMP_GT, PS_SELF},     {"int3211", P_DF, P_PP, CMP_GT, PS_SELF},
    {"int3220", P_DF, P_SD, CMP_GT, PS_SELF},     {"int3221", P_DF, P_PD, CMP_GT, PS_SELF},
    {"int3222", P_DF, P_DD, CMP_GT, PS_SELF},     {"int3230", P_DF, P_SF, CMP_GT, PS_SELF},
    {"int3231", P_DF, P_PF, CMP_GT, PS_SELF},     {"int3232", P_DF, P_DF, CMP_GT, PS_SELF},
    {"int3300", P_FF, P_SS, CMP_GT, PS_SELF},     {"int3310", P_FF, P_SP, CMP_GT, PS_SELF},
    {"int3311", P_FF, P_PP, CMP_GT, PS_SELF},     {"int3320", P_FF, P_SD, CMP_GT, PS_SELF},
    {"int3321", P_FF, P_PD, CMP_GT, PS_SELF},     {"int3322", P_FF, P_DD, CMP_GT, PS_SELF},
    {"int3332", P_FF, P_DF, CMP_GT, PS_SELF},
};

}  // namespace liberi

using namespace liberi;

// ------------------------------------------------------------------ errors
static thread_local std::string g_last_error;

static int fail(int code, const std::string &msg) {
  g_last_error = msg;
  return code;
}

#define HIP_TRY(expr)                                                                                   \
  do {                                                                                                  \
    hipError_t e_ = (expr);                                                                             \
    if (e_ != hipSuccess)                                                                               \
      return fail(e_ == hipErrorOutOfMemory ? LIBERI_ENOMEM : LIBERI_EDEVICE,                           \
                  std::string(#expr) + ": " + hipGetErrorString(e_));                                   \
  } while (0)

static void forget_tuned_choices();

// --------------------------------------------------------------- handle
struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
};

struct ClassState {
  bool active = false;
  bool row_ok = false;  // a row-tiled kernel exists and fits in LDS
  int variant = -1;     // form chosen for the class: 0 direct, 1 row-tiled, 3 cooperative (-1: not yet)
  int fp32 = -1;        // mixed form: 1 FP32 allowed, 0 not (-1: not yet chosen for the current tau)
  float ms = -1.f;      // device time of the class's launch, measured at the first build
  int64_t nquart = 0, nprimq = 0;
  int32_t nseg = 0;
  int tile = -1;        // row tiles chosen for the class, index into `tiles` (-1: not yet)
  // the row tiles of this rank's share, for each tile length and, for a class of
  // few quartets (`small`), of one workgroup step each (kStepTile)
  const RowTile *tiles[kNumTileLens + 1] = {};
  int32_t ntile[kNumTileLens + 1] = {};
  bool small = false;
  ClassDev dev{};
  // form of the last build, as in liberi_stats (-1: not built)
  int32_t ran = -1, ran_tile = 0, ran_fp32 = 0;
  // shared launch the class has a place in (-1: none), its workgroups there and,
  // in a row-tiled one, its tiles; the choices above are those of its own launch
  int shared = -1;
  int32_t shared_groups = 0;
  const RowTile *shared_tiles = nullptr;
};

// index of the tiles of one workgroup step
constexpr int kStepTile = kNumTileLens;

// the row tiles where none are timed or asked for
static int default_tile(const ClassState &cs_) { return cs_.small ? kStepTile : kDefaultTile; }

// length of tiles k of class c
static int64_t tile_length(int c, int k) { return k == kStepTile ? class_row_quartets(c) : kTileLens[k]; }

// Point the class's launch arguments at its row tiles k.
static void use_tiles(ClassState &cs_, int k) {
  cs_.dev.tiles = cs_.tiles[k];
  cs_.dev.ntile = cs_.ntile[k];
}

struct liberi_ctx {
  // options
  double schwarz_cut = kRefCutoff, value_cut = kRefCutoff, fp32_tau = 0.0, exact_large_t = 0.0;
  double prim_cut = 1e-18;
  int row_tiles = 1;  // 0 never, 1 per class (autotuned or default), 2 wherever they fit
  bool autotune = true;
  double max_device_bytes = 0.0;  // HBM budget of the handle (0: none)
  int rank_split = 0;             // 0 shares balanced by estimated cost, 1 equal quartet counts
  // basis
  bool initialized = false;
  int32_t nsh = 0, natoms = 0, num_bas = 0, mxgtot = 0, rank = 0, nprocs = 1;
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // builds share the handle's workspace (Dp, Jp, Dsq): each waits for the end
  // of the last one, on whatever stream that was.  ev1 is that end (built: it
  // has been recorded); a build under a caller's capture, which does not run
  // then, records neither event.
  bool built = false;
  // the end of every kPace-th build, in turn: at most 2 kPace are outstanding
  hipEvent_t paced[2] = {};
  bool paced_set[2] = {};
  int pace_slot = 0, pace_count = 0;
  std::vector<DevBuf> owned;
  DevBuf pairs, prims, dens, fock;
  DevBuf tables;  // segments and row tiles of every class
  PairLayout layout{};      // pair layout of the basis
  // per build: density and Coulomb sums by pair (component- then pair-major),
  // square exchange density and exchange sums
  DevBuf dpair, jpair, dsq, ksq;
  DevBuf col_bf[4];     // compact columns per angular momentum -> basis function
  int32_t ncol[4] = {};
  DevBuf aux;           // per build: max |D|, FP32 quartet count
  // fused group launch: work items, every class's ClassDev, the queue head
  DevBuf fused_items, fused_cds, fused_head;
  int64_t fused_n = 0;
  int fused_nwg = 0;
  // shared launches of small classes and the ClassDev of every class in them
  SharedArgs shared[kSharedLaunches];
  DevBuf shared_cds;
  bool fused = false;      // LIBERI_OPT_FUSED
  int row_orient = 0;      // LIBERI_OPT_ROW_ORIENT
  int tile_len = -1;       // LIBERI_OPT_TILE_LEN as an index into kTileLens; -1 chosen per class
  DevBuf tune_F;        // autotuner's scratch Fock matrix
  DevBuf dens_t, dens_b, fock_b;  // UHF: Da + Db, and the beta density / Fock of the host entry point
  hipEvent_t tev[2] = {};
  // batched form: the build's class launches spread over the branches of a
  // graph, captured once and replayed by later builds on the same D and F
  bool use_graph = true;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  const double *g_dD = nullptr;
  double *g_dF = nullptr;
  // the same for the two builds of an unrestricted one: the graph, the arrays
  // (Da, Db, Fa, Fb) it was captured with and those of the last call, and the
  // second build's workspace
  hipGraph_t ugraph = nullptr;
  hipGraphExec_t uexec = nullptr;
  const void *ug_arrays[4] = {}, *u_arrays[4] = {};
  DevBuf uhf_work;
  // workspaces of the builds in graphs of the caller's, one per Fock array: two
  // builds into one array cannot run side by side anyway, those into others
  // may, and beside the builds of the handle
  std::vector<std::pair<const double *, DevBuf>> captured;
  bool uhf_refused = false;  // no memory for it: the spins' builds run one after the other
  bool fp32_pending = false;
  ClassState cls[kNumClasses];
  liberi_stats stats{};
  // diagnostics
  bool class_timing = false, timing_pending = false, build_pending = false;
  int only_class = -1;
  hipEvent_t cev0[kNumClasses] = {}, cev1[kNumClasses] = {};
};

// fold the events of the last build into the statistics (waits for it)
static void collect_timing(liberi_ctx *h) {
  if (h->build_pending) {
    if (h->built && hipEventSynchronize(h->ev1) == hipSuccess) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, h->ev0, h->ev1) == hipSuccess) h->stats.last_build_ms = ms;
    }
    h->build_pending = false;
    if (h->fp32_pending) {
      uint64_t n = 0;
      if (hipMemcpy(&n, (uint64_t *)h->aux.p + 1, sizeof(n), hipMemcpyDeviceToHost) == hipSuccess)
        h->stats.fp32_quartets = (int64_t)n;
      h->fp32_pending = false;
    }
  }
  if (!h->timing_pending) return;
  for (int c = 0; c < kNumClasses; ++c) {
    h->stats.class_ms[c] = 0.0;
    if (!h->cls[c].active || !h->cev0[c]) continue;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, h->cev0[c], h->cev1[c]) == hipSuccess) h->stats.class_ms[c] = ms;
  }
  h->timing_pending = false;
}

// bytes of HBM counted as held by the handle, within its budget
static int charge(liberi_ctx *h, size_t bytes) {
  if (h->max_device_bytes > 0.0 && (double)h->stats.device_bytes + (double)bytes > h->max_device_bytes)
    return fail(LIBERI_ENOMEM, "device budget of the handle (LIBERI_OPT_MAX_DEVICE_BYTES = " +
                                   std::to_string((int64_t)h->max_device_bytes) + ") exceeded by an allocation of " +
                                   std::to_string(bytes) + " bytes");
  h->stats.device_bytes += (int64_t)bytes;
  return LIBERI_OK;
}

// an allocation whose bytes are already charged
static int dev_alloc_charged(DevBuf &b, size_t bytes) {
  b = DevBuf{};
  if (bytes == 0) return LIBERI_OK;
  const hipError_t e = hipMalloc(&b.p, bytes);
  if (e != hipSuccess) {
    // (a caller may go on without the memory: the launches after it return the
    // thread's last error, which later successful calls leave as it is)
    (void)hipGetLastError();
    b.p = nullptr;
    return fail(e == hipErrorOutOfMemory ? LIBERI_ENOMEM : LIBERI_EDEVICE,
                "hipMalloc(" + std::to_string(bytes) + "): " + hipGetErrorString(e));
  }
  b.bytes = bytes;
  return LIBERI_OK;
}

static int dev_alloc(liberi_ctx *h, DevBuf &b, size_t bytes) {
  b = DevBuf{};
  if (bytes == 0) return LIBERI_OK;
  if (int rc = charge(h, bytes)) return rc;
  const int rc = dev_alloc_charged(b, bytes);
  if (rc) h->stats.device_bytes -= (int64_t)bytes;
  return rc;
}

template <class T>
static int dev_upload(liberi_ctx *h, DevBuf &b, const std::vector<T> &v) {
  int rc = dev_alloc(h, b, v.size() * sizeof(T));
  if (rc) return rc;
  if (!v.empty()) HIP_TRY(hipMemcpy(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return LIBERI_OK;
}

static void dev_free(DevBuf &b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.bytes = 0;
}

// Waits on the host for an event of builds that run (a thread that captures
// may call it: it waits for nothing captured).
static hipError_t wait_event(hipEvent_t e) {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  const hipError_t rc = hipEventSynchronize(e);
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  return rc;
}

// Waits on the host for the last build that ran, on whatever stream.
static void wait_last_build(liberi_ctx *h) {
  if (h->built) (void)wait_event(h->ev1);
}

// The end of a build on st.  A caller that enqueues builds without ever
// waiting gets ahead of the device without bound, thousands of graph launches
// for a small molecule; here it waits for the build kPace to 2 kPace before, so
// that the device always has some to go on with.
constexpr int kPace = 8;
static hipError_t end_build(liberi_ctx *h, hipStream_t st) {
  hipError_t e = hipEventRecord(h->ev1, st);
  if (e != hipSuccess) return e;
  h->built = true;
  if (++h->pace_count < kPace) return hipSuccess;
  h->pace_count = 0;
  const int k = h->pace_slot;
  if ((e = hipEventRecord(h->paced[k], st)) != hipSuccess) return e;
  h->paced_set[k] = true;
  h->pace_slot = k ^ 1;
  return h->paced_set[k ^ 1] ? wait_event(h->paced[k ^ 1]) : hipSuccess;
}

// A graph taken from the handle, destroyed once its replays are over.
struct OldGraph {
  liberi_ctx *h;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  OldGraph(liberi_ctx *h_, hipGraph_t &g, hipGraphExec_t &e) : h(h_) {
    std::swap(graph, g);
    std::swap(exec, e);
  }
  OldGraph(const OldGraph &) = delete;
  OldGraph &operator=(const OldGraph &) = delete;
  ~OldGraph() { end(); }
  void end() {
    if (exec) {
      wait_last_build(h);
      (void)hipGraphExecDestroy(exec);
    }
    if (graph) (void)hipGraphDestroy(graph);
    exec = nullptr;
    graph = nullptr;
  }
};

static void drop_graph(liberi_ctx *h) {
  OldGraph(h, h->ugraph, h->uexec);
  OldGraph(h, h->graph, h->gexec);
  h->g_dD = nullptr;
  h->g_dF = nullptr;
}

static void release_device(liberi_ctx *h) {
  wait_last_build(h);
  drop_graph(h);
  std::fill(h->u_arrays, h->u_arrays + 4, nullptr);
  dev_free(h->uhf_work);
  h->uhf_refused = false;
  for (auto &w : h->captured) dev_free(w.second);
  h->captured.clear();
  for (auto &c : h->cls) {
    c = ClassState{};
  }
  dev_free(h->tables);
  dev_free(h->pairs);
  dev_free(h->prims);
  dev_free(h->dens);
  dev_free(h->fock);
  dev_free(h->aux);
  for (auto &sa : h->shared) sa = SharedArgs{};
  dev_free(h->shared_cds);
  dev_free(h->fused_items);
  dev_free(h->fused_cds);
  dev_free(h->fused_head);
  h->fused_n = 0;
  dev_free(h->tune_F);
  dev_free(h->dpair);
  dev_free(h->jpair);
  dev_free(h->dsq);
  dev_free(h->ksq);
  dev_free(h->dens_t);
  dev_free(h->dens_b);
  dev_free(h->fock_b);
  for (auto &b : h->col_bf) dev_free(b);
  for (auto &n : h->ncol) n = 0;
  // (nothing is left of the last build to report: its counter is gone)
  h->build_pending = h->fp32_pending = h->timing_pending = false;
  h->stats = liberi_stats{};
  h->initialized = false;
}

extern "C" {

const char *liberi_c_last_error(void) { return g_last_error.c_str(); }

const char *liberi_c_class_name(int32_t c) { return (c >= 0 && c < kNumClasses) ? kClasses[c].name : ""; }

// Kernel attributes of every class, once per device in the process, at
// handle creation (never inside a stream capture)
static int prepare_kernels(int device) {
  static std::mutex mu;
  static std::vector<int> done;
  std::lock_guard<std::mutex> lk(mu);
  if (std::find(done.begin(), done.end(), device) != done.end()) return LIBERI_OK;
  for (int c = 0; c < kNumClasses; ++c)
    if (int e = prepare_class(c))
      return fail(LIBERI_EDEVICE, std::string("kernel attributes of ") + kClasses[c].name + ": " +
                                      hipGetErrorString((hipError_t)e));
  done.push_back(device);
  return LIBERI_OK;
}

int liberi_c_create(liberi_ctx **ctx) {
  if (!ctx) return fail(LIBERI_EARG, "liberi_c_create: NULL handle pointer");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return fail(LIBERI_EDEVICE, "liberi_c_create: no HIP device visible");
  auto *h = new (std::nothrow) liberi_ctx();
  if (!h) return fail(LIBERI_ENOMEM, "liberi_c_create: out of host memory");
  HIP_TRY(hipGetDevice(&h->device));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, h->device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    delete h;
    return fail(LIBERI_EDEVICE, std::string("liberi_c_create: device is ") + prop.gcnArchName +
                                    ", this library is built for gfx950 (MI355X)");
  }
  if (int rc = prepare_kernels(h->device)) {
    delete h;
    return rc;
  }
  HIP_TRY(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  HIP_TRY(hipEventCreate(&h->ev0));
  HIP_TRY(hipEventCreate(&h->ev1));
  for (hipEvent_t &e : h->paced) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  *ctx = h;
  return LIBERI_OK;
}

int liberi_c_cleanup(liberi_ctx *h) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_cleanup: NULL handle");
  // not set up: nothing to do (src/interface/liberi_interface.F90:235), but
  // device data of a setup that failed part of the way is released as well
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  release_device(h);
  return LIBERI_OK;
}

int liberi_c_destroy(liberi_ctx **ctx) {
  if (!ctx) return fail(LIBERI_EARG, "liberi_c_destroy: NULL handle pointer");
  liberi_ctx *h = *ctx;
  if (!h) return LIBERI_OK;
  liberi_c_cleanup(h);
  if (h->ev0) (void)hipEventDestroy(h->ev0);
  if (h->ev1) (void)hipEventDestroy(h->ev1);
  for (hipEvent_t e : h->tev)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : h->paced)
    if (e) (void)hipEventDestroy(e);
  for (int c = 0; c < kNumClasses; ++c) {
    if (h->cev0[c]) (void)hipEventDestroy(h->cev0[c]);
    if (h->cev1[c]) (void)hipEventDestroy(h->cev1[c]);
  }
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  *ctx = nullptr;
  return LIBERI_OK;
}

int liberi_c_set_option(liberi_ctx *h, int32_t opt, double v) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_set_option: NULL handle");
  drop_graph(h);  // a captured build holds the options it was captured with
  if (opt == LIBERI_OPT_ONLY_CLASS) {
    if (!(v >= -1.0 && v < kNumClasses) || v != std::floor(v))
      return fail(LIBERI_EARG, "liberi_c_set_option: ONLY_CLASS must be -1 or a class index 0..54");
    h->only_class = (int)v;
    return LIBERI_OK;
  }
  if (!(v >= 0.0) || !std::isfinite(v)) return fail(LIBERI_EARG, "liberi_c_set_option: value must be finite, >= 0");
  switch (opt) {
    case LIBERI_OPT_CLASS_TIMING: h->class_timing = v != 0.0; break;
    case LIBERI_OPT_SCHWARZ_CUTOFF: h->schwarz_cut = v; break;
    case LIBERI_OPT_VALUE_CUTOFF: h->value_cut = v; break;
    case LIBERI_OPT_FP32_TAU:
      if (v != h->fp32_tau)
        for (auto &c : h->cls) c.fp32 = -1;  // chosen again at the next build
      h->fp32_tau = v;
      break;
    case LIBERI_OPT_EXACT_LARGE_T: h->exact_large_t = v != 0.0; break;
    case LIBERI_OPT_PRIM_CUTOFF: h->prim_cut = v; break;
    case LIBERI_OPT_ROW_TILES:
      if (v != 0.0 && v != 1.0 && v != 2.0) return fail(LIBERI_EARG, "liberi_c_set_option: ROW_TILES must be 0, 1 or 2");
      h->row_tiles = (int)v;
      break;
    case LIBERI_OPT_GRAPH: h->use_graph = v != 0.0; break;
    case LIBERI_OPT_MAX_DEVICE_BYTES:
      h->max_device_bytes = v;
      h->uhf_refused = false;
      break;
    case LIBERI_OPT_RANK_SPLIT:
      if (v != 0.0 && v != 1.0) return fail(LIBERI_EARG, "liberi_c_set_option: RANK_SPLIT must be 0 or 1");
      h->rank_split = (int)v;
      break;
    case LIBERI_OPT_FUSED: h->fused = v != 0.0; break;
    case LIBERI_OPT_ROW_ORIENT:
      if (v != 0.0 && v != 1.0 && v != 2.0) return fail(LIBERI_EARG, "liberi_c_set_option: ROW_ORIENT must be 0, 1 or 2");
      h->row_orient = (int)v;
      break;
    case LIBERI_OPT_TILE_LEN: {
      int k = -1;
      for (int i = 0; i < kNumTileLens; ++i)
        if (v == (double)kTileLens[i]) k = i;
      if (v != 0.0 && k < 0)
        return fail(LIBERI_EARG, "liberi_c_set_option: TILE_LEN must be 0, 512, 1024, 4096 or 16384");
      h->tile_len = v == 0.0 ? -1 : k;
      for (auto &c : h->cls) c.tile = -1;  // chosen again at the next build
      break;
    }
    case LIBERI_OPT_AUTOTUNE:
      h->autotune = v != 0.0;
      // decide (and time) again at the next build, without earlier handles' choices
      for (auto &c : h->cls) c.variant = -1, c.fp32 = -1, c.tile = -1, c.ms = -1.f;
      forget_tuned_choices();
      break;
    default: return fail(LIBERI_EARG, "liberi_c_set_option: unknown option " + std::to_string(opt));
  }
  return LIBERI_OK;
}

int liberi_c_get_option(liberi_ctx *h, int32_t opt, double *v) {
  if (!h || !v) return fail(LIBERI_EARG, "liberi_c_get_option: NULL argument");
  switch (opt) {
    case LIBERI_OPT_SCHWARZ_CUTOFF: *v = h->schwarz_cut; break;
    case LIBERI_OPT_VALUE_CUTOFF: *v = h->value_cut; break;
    case LIBERI_OPT_FP32_TAU: *v = h->fp32_tau; break;
    case LIBERI_OPT_EXACT_LARGE_T: *v = h->exact_large_t; break;
    case LIBERI_OPT_PRIM_CUTOFF: *v = h->prim_cut; break;
    case LIBERI_OPT_CLASS_TIMING: *v = h->class_timing; break;
    case LIBERI_OPT_ONLY_CLASS: *v = h->only_class; break;
    case LIBERI_OPT_ROW_TILES: *v = h->row_tiles; break;
    case LIBERI_OPT_AUTOTUNE: *v = h->autotune; break;
    case LIBERI_OPT_GRAPH: *v = h->use_graph; break;
    case LIBERI_OPT_MAX_DEVICE_BYTES: *v = h->max_device_bytes; break;
    case LIBERI_OPT_RANK_SPLIT: *v = h->rank_split; break;
    case LIBERI_OPT_FUSED: *v = h->fused; break;
    case LIBERI_OPT_ROW_ORIENT: *v = h->row_orient; break;
    case LIBERI_OPT_TILE_LEN: *v = h->tile_len < 0 ? 0.0 : (double)kTileLens[h->tile_len]; break;
    default: return fail(LIBERI_EARG, "liberi_c_get_option: unknown option " + std::to_string(opt));
  }
  return LIBERI_OK;
}

int liberi_c_get_stats(liberi_ctx *h, liberi_stats *out) {
  if (!h || !out) return fail(LIBERI_EARG, "liberi_c_get_stats: NULL argument");
  collect_timing(h);
  *out = h->stats;
  for (int c = 0; c < kNumClasses; ++c) {
    out->class_variant[c] = h->cls[c].ran;
    out->class_fp32[c] = h->cls[c].ran_fp32;
    out->class_tile[c] = h->cls[c].ran_tile;
  }
  return LIBERI_OK;
}

// ------------------------------------------------------------------ setup
// Where the reference stops using its tabulated Boys function / Rys roots.
// Rotated-axis and ERIC kernels (classes 0-13 and 22-25) take the asymptotic
// Boys chain F_m = F_{m-1} (2m-1)/2T for T > t_max = 25
// (src/liberi_boys.F90:22, src/rhf/rot_axis/int1111.F90:389-396,
// src/rhf/eric/int0030_ericgen.F90:300-311); the Rys kernels take the
// asymptotic roots for X >= 37, 43, 49, 55, 60, 65 with 2..7 roots
// (e.g. src/rhf/rot_axis/int2222_rysgen.F90:642).  Switching the Rys rule at
// the same points reproduces those values.
static double reference_switch(int c) {
  if (c <= 13 || (c >= 22 && c <= 25)) return std::nextafter(25.0, INFINITY);  // table iff T <= 25
  static const double thr[8] = {0, 0, 37.0, 43.0, 49.0, 55.0, 60.0, 65.0};       // table iff X < thr
  return thr[class_nroots(c)];
}

struct HostShell {
  int l, k, bf0;
  double c[3];
  const double *e, *w;
};

// Shells from the reference's setup arrays (src/liberi_shell_pair.F90:108-135),
// with the argument checks the reference leaves to the caller.
static int read_shells(const char *who, int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                       const int32_t *ang_mom, const int32_t *contr_num, const int32_t *sh_loc,
                       const int32_t *atom_num, const int32_t *atom_loc, const double *exponents, const double *cs,
                       const double *cp, const double *cdc, const double *cf, const double *coords,
                       std::vector<HostShell> &sh) {
  const std::string w0 = std::string(who) + ": ";
  if (nsh <= 0 || natoms <= 0 || num_bas <= 0 || mxgtot <= 0)
    return fail(LIBERI_EARG, w0 + "nsh, natoms, num_bas, mxgtot must be positive");
  // the packed matrices hold num_bas(num_bas+1)/2 elements, a default
  // integer in the reference's interface (liberi_interface.F90:202-217);
  // the kernels index them in 32 bits
  if (num_bas > kMaxBasis)
    return fail(LIBERI_EARG, w0 + "num_bas above " + std::to_string(kMaxBasis) + " (packed size exceeds 32 bits)");
  if (!ang_mom || !contr_num || !sh_loc || !atom_num || !atom_loc || !exponents || !cs || !cp || !cdc || !cf ||
      !coords)
    return fail(LIBERI_EARG, w0 + "NULL array");
  sh.assign(nsh, HostShell{});
  const int64_t coef_len = (int64_t)mxgtot * nsh;
  for (int s = 0; s < nsh; ++s) {
    const int l = ang_mom[s] - 1, k = contr_num[s], loc = sh_loc[s] - 1, a = atom_num[s] - 1;
    if (l < 0 || l > 3) return fail(LIBERI_EARG, w0 + "ang_mom must be 1..4 (shell " + std::to_string(s + 1) + ")");
    if (k < 1 || loc < 0 || loc + k > coef_len)
      return fail(LIBERI_EARG, w0 + "contr_num/sh_loc out of range (shell " + std::to_string(s + 1) + ")");
    if (a < 0 || a >= natoms) return fail(LIBERI_EARG, w0 + "atom_num out of range");
    const int bf0 = atom_loc[s] - 1;
    if (bf0 < 0 || bf0 + (l + 1) * (l + 2) / 2 > num_bas) return fail(LIBERI_EARG, w0 + "atom_loc out of range");
    const double *w = l == 0 ? cs : l == 1 ? cp : l == 2 ? cdc : cf;
    for (int i = 0; i < k; ++i)
      if (!(exponents[loc + i] > 0.0) || !std::isfinite(exponents[loc + i]) || !std::isfinite(w[loc + i]))
        return fail(LIBERI_EARG, w0 + "exponents must be finite and > 0, coefficients finite (shell " +
                                     std::to_string(s + 1) + ")");
    sh[s] = HostShell{l, k, bf0, {coords[3 * a], coords[3 * a + 1], coords[3 * a + 2]}, exponents + loc, w + loc};
  }
  return LIBERI_OK;
}

static int ncart_host(int l) { return (l + 1) * (l + 2) / 2; }

// Shell pair (sA, sB) and its primitive pairs appended to the device records
// (the per-primitive-pair quantities of src/liberi_shell_pair.F90:416-459);
// rank[s] = position of shell s among the shells of its angular momentum.
static void append_pair(std::vector<PairRec> &pairs, std::vector<PrimRec> &prims, const std::vector<HostShell> &sh,
                        const std::vector<int> &rank, int sA, int sB) {
  const HostShell &A = sh[sA], &B = sh[sB];
  PairRec r{};
  r.prim_off = (int32_t)prims.size();
  r.nprim = A.k * B.k;
  r.bfA = A.bf0;
  r.bfB = B.bf0;
  r.ABx = A.c[0] - B.c[0];
  r.ABy = A.c[1] - B.c[1];
  r.ABz = A.c[2] - B.c[2];
  r.sameAB = sA == sB;
  r.prim_stride = 1;
  r.cA = rank[sA] * ncart_host(A.l);
  r.cB = rank[sB] * ncart_host(B.l);
  const double ab2 = r.ABx * r.ABx + r.ABy * r.ABy + r.ABz * r.ABz;
  for (int i = 0; i < A.k; ++i)
    for (int j = 0; j < B.k; ++j) {
      const double a = A.e[i], b = B.e[j], p = a + b;
      PrimRec pr;
      pr.p = p;
      pr.Px = (a * A.c[0] + b * B.c[0]) / p;
      pr.Py = (a * A.c[1] + b * B.c[1]) / p;
      pr.Pz = (a * A.c[2] + b * B.c[2]) / p;
      pr.PAx = pr.Px - A.c[0];
      pr.PAy = pr.Py - A.c[1];
      pr.PAz = pr.Pz - A.c[2];
      pr.K = A.w[i] * B.w[j] * std::exp(-a * b / p * ab2) / p;
      prims.push_back(pr);
    }
  pairs.push_back(r);
}

// Work items of the fused group launch: every active class that has a body
// in it, in runs of kFusedRounds rounds of its quartets per item; the classes
// in order of their primitive quartets (largest first), the items of a class
// dealt out over its whole quartet range (item k takes run k x stride mod n,
// stride coprime with n) so that the workgroups running at the same time
// meet few common Fock rows.
constexpr int64_t kFusedRounds = 32;

// Classes of at most this many workgroups run in a shared launch: row tiles
// of 256 lanes, and waves of the group and cooperative forms.  Larger classes
// fill the chip by themselves, and in a shared launch they would run at the
// registers of its largest class (12 atoms of the cage: 1024 / 4096 1.08 ms,
// 2048 / 4096 1.10, 8192 / 32768 1.24; unrestricted 17-atom cluster 1.06, 0.97,
// 0.98 ms; 41-atom cluster 5.24, 5.31, 5.40).
constexpr int64_t kSharedRowGroups = 2048, kSharedWaveGroups = 4096;

static int setup_fused(liberi_ctx *h) {
  std::vector<int> cls;
  for (int c = 0; c < kNumClasses; ++c)
    if (h->cls[c].active && class_fused_nq(c) > 0 && h->cls[c].dev.q_end > h->cls[c].dev.q_begin) cls.push_back(c);
  h->fused_n = 0;
  if (cls.empty()) return LIBERI_OK;
  std::stable_sort(cls.begin(), cls.end(), [&](int a, int b) { return h->cls[a].nprimq > h->cls[b].nprimq; });
  std::vector<FusedItem> items;
  for (int c : cls) {
    const ClassDev &d = h->cls[c].dev;
    const int64_t nq = d.q_end - d.q_begin, run = kFusedRounds * class_fused_nq(c);
    const int64_t n = (nq + run - 1) / run, stride = chunk_stride(n);
    for (int64_t k = 0; k < n; ++k) {
      const int64_t j = k * stride % n;
      items.push_back(FusedItem{c, 0, j * run, std::min(nq, (j + 1) * run)});
    }
  }
  std::vector<ClassDev> cds(kNumClasses);
  for (int c = 0; c < kNumClasses; ++c) cds[c] = h->cls[c].dev;
  int rc;
  if ((rc = dev_upload(h, h->fused_items, items)) || (rc = dev_upload(h, h->fused_cds, cds)) ||
      (rc = dev_alloc(h, h->fused_head, sizeof(double))))
    return rc;
  int ncu = 0;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device) != hipSuccess || ncu <= 0) ncu = 256;
  h->fused_nwg = 12 * ncu;  // three one-wave workgroups per SIMD
  h->fused_n = (int64_t)items.size();
  return LIBERI_OK;
}

// Proxy for the device time of class c (ms): primitive quartets x Rys roots x
// sqrt(cartesian components).
static double class_cost_proxy(const liberi_ctx *h, int c) {
  const int la = kPairL[kClasses[c].bra][1], lb = kPairL[kClasses[c].bra][0];
  const int lc = kPairL[kClasses[c].ket][1], ld = kPairL[kClasses[c].ket][0];
  const double ncomp = (double)ncart_host(la) * ncart_host(lb) * ncart_host(lc) * ncart_host(ld);
  return 1e-9 * (double)h->cls[c].nprimq * class_nroots(c) * std::sqrt(ncomp);
}

// The shared launches: of the classes with a place in one, those that do not
// have it to themselves; the class with the longest workgroups first.
static int setup_shared(liberi_ctx *h) {
  std::vector<ClassDev> cds(kNumClasses);
  for (int k = 0; k < kSharedLaunches; ++k) {
    SharedArgs &sa = h->shared[k] = SharedArgs{};
    std::vector<int> cls;
    for (int c = 0; c < kNumClasses; ++c)
      if (h->cls[c].shared == k) cls.push_back(c);
    if (cls.size() < 2) {
      for (int c : cls) h->cls[c].shared = -1;
      continue;
    }
    auto per_group = [&](int c) { return class_cost_proxy(h, c) / h->cls[c].shared_groups; };
    std::stable_sort(cls.begin(), cls.end(), [&](int a, int b) { return per_group(a) > per_group(b); });
    int64_t at = 0;
    for (int c : cls) {
      ClassState &cs_ = h->cls[c];
      ClassDev &d = cds[c] = cs_.dev;
      d.tiles = cs_.shared_tiles;
      d.ntile = cs_.shared_groups;
      d.chunk_stride = chunk_stride(cs_.shared_groups);
      d.fp32 = 0;
      if (k < kSharedRowLaunches)
        sa.lds = std::max(sa.lds, (int32_t)class_row_lds(c, d.transposed, h->ncol, d.xswitch));
      sa.cls[sa.n] = c;
      sa.first[sa.n++] = (int32_t)at;
      at += cs_.shared_groups;
      sa.first[sa.n] = (int32_t)at;
    }
  }
  return dev_upload(h, h->shared_cds, cds);
}

// Row tiles of the quartets [q_begin, q_end) of class c, in launch order: the
// rows of the fixed pairs with the most primitives first (the kept rows run
// from few to many), the longest rows first among those.  Consecutive
// segments of a row whose quartets are shared by the same number of lanes are
// cut into tiles of `len` quartets at one lane each, fewer at more.  `cut`: some
// were longer, so that a larger `len` gives other tiles.
static std::vector<RowTile> row_tiles(int c, int64_t q_begin, int64_t q_end, int64_t primq, int64_t len, bool &cut,
                                      const std::vector<int64_t> &sstart, const std::vector<int32_t> &sbra,
                                      const std::vector<int32_t> &sket0, const std::vector<PairRec> &pairs) {
  std::vector<RowTile> tiles;
  cut = false;
  if (q_begin >= q_end) return tiles;
  const size_t s0 = (size_t)(std::upper_bound(sstart.begin(), sstart.end(), q_begin) - sstart.begin()) - 1;
  const size_t s1 = (size_t)(std::lower_bound(sstart.begin(), sstart.end(), q_end) - sstart.begin());
  // rows [first segment, last) of the share
  std::vector<std::pair<size_t, size_t>> rows;
  for (size_t a = s0, b; a < s1; a = b) {
    for (b = a; b < s1 && sbra[b] == sbra[a];) ++b;
    rows.push_back({a, b});
  }
  const double chain = class_row_chain(c, primq);
  auto team_of = [&](size_t s) {
    int32_t t = 1;
    if (chain > 0.0) {
      const int nf = pairs[sbra[s]].nprim, nm = pairs[sket0[s]].nprim;
      while (t < 64 && t < nm && (double)((nm + t - 1) / t) * nf > chain) t *= 2;
      while (t > 1 && (nm + t / 2 - 1) / (t / 2) == (nm + t - 1) / t) t /= 2;  // no shorter chain
    }
    return t;
  };
  auto cut_row = [&](size_t a, size_t b) {
    for (size_t s = a, e; s < b; s = e) {
      const int32_t team = team_of(s);
      for (e = s + 1; e < b && team_of(e) == team;) ++e;
      const int64_t cap = std::max<int64_t>(1, len / team);
      size_t sg = s;
      const int64_t q1 = std::min(sstart[e], q_end), qs = std::max(sstart[s], q_begin);
      cut |= q1 - qs > cap;
      for (int64_t q = qs; q < q1; q += cap) {
        while (sstart[sg + 1] <= q) ++sg;
        const int64_t n = std::min(cap, q1 - q);
        size_t last = sg;
        while (sstart[last + 1] < q + n) ++last;
        tiles.push_back(RowTile{q, (int32_t)n, (int32_t)sg, team, (int32_t)last});
      }
    }
  };
  for (size_t hi = rows.size(); hi > 0;) {
    size_t lo = hi - 1;
    auto np = [&](size_t r) { return pairs[sbra[rows[r].first]].nprim; };
    while (lo > 0 && np(lo - 1) == np(hi - 1)) --lo;
    for (size_t r = lo; r < hi; ++r) cut_row(rows[r].first, rows[r].second);
    hi = lo;
  }
  return tiles;
}

// Setup proper, on a handle whose device data is released; the caller
// releases whatever it leaves behind when it fails part of the way through.
static int setup_basis(liberi_ctx *h, int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                       const std::vector<HostShell> &sh, const double *schwrz, int32_t my_rank, int32_t num_procs) {
  h->nsh = nsh;
  h->natoms = natoms;
  h->num_bas = num_bas;
  h->mxgtot = mxgtot;
  h->rank = my_rank;
  h->nprocs = num_procs;

  // ---- shell lists per L, ascending index (src/liberi_shell_pair.F90:137-344)
  std::vector<int> lists[4];
  for (int s = 0; s < nsh; ++s) lists[sh[s].l].push_back(s);
  // compact columns: the functions of each angular momentum in shell order
  std::vector<int> rank(nsh);
  {
    std::vector<int32_t> cols[4];
    for (int l = 0; l < 4; ++l) {
      for (size_t k = 0; k < lists[l].size(); ++k) {
        rank[lists[l][k]] = (int)k;
        for (int m = 0; m < ncart_host(l); ++m) cols[l].push_back(sh[lists[l][k]].bf0 + m);
      }
      h->ncol[l] = (int32_t)cols[l].size();
      if (int rc1 = dev_upload(h, h->col_bf[l], cols[l])) return rc1;
    }
  }

  // ---- pair classes: records, Schwarz values (compute_*_pairs, :348-1682)
  std::vector<PairRec> pairs;
  std::vector<PrimRec> prims;
  std::vector<double> pair_x;
  std::vector<std::vector<int32_t>> class_pairs(kNumPairClasses);
  auto add_pair = [&](int pc, int sA, int sB) {
    const int hi = std::max(sA, sB), lo = std::min(sA, sB);
    pair_x.push_back(schwrz[(int64_t)hi * (hi + 1) / 2 + lo]);
    class_pairs[pc].push_back((int32_t)pairs.size());
    append_pair(pairs, prims, sh, rank, sA, sB);
    pairs.back().x = pair_x.back();
  };
  for (int pc = 0; pc < kNumPairClasses; ++pc) {
    const int l1 = kPairL[pc][0], l2 = kPairL[pc][1];
    if (l1 == l2) {
      for (size_t ii = 0; ii < lists[l1].size(); ++ii)
        for (size_t jj = 0; jj <= ii; ++jj) add_pair(pc, lists[l1][ii], lists[l1][jj]);
    } else {
      for (int x : lists[l1])
        for (int y : lists[l2]) add_pair(pc, y, x);  // A = the higher-L shell
    }
  }
  if (prims.size() > (size_t)INT32_MAX || pairs.size() > (size_t)INT32_MAX)
    return fail(LIBERI_EARG, "liberi_c_setup: basis too large for 32-bit pair indices");

  // ---- primitive-pair screen.  Bound of one primitive pair's share of any
  // integral: B = 2pi^(5/2)^(1/2) |K| (1 + |P-A| + 1/sqrt(p))^(la+lb) (the
  // Rys 2-D factors are polynomials in P-A, P-Q and 1/2p of that degree, the
  // Boys values are <= 1); a primitive quartet contributes at most about
  // B_ab B_cd.  A primitive pair of shell pair ab only ever meets the
  // primitive pairs of ab's partners: the shell pairs cd with
  // x_ab x_cd >= cutoff (every quartet test compares that product), and every
  // pair of the other list in the classes without a quartet test.  With M_ab
  // the largest B among those partners, primitive pairs with B M_ab <
  // prim_cut change no integral by more than prim_cut per primitive quartet,
  // far below the value cutoff, and are dropped.  Quartet lists and counts are
  // untouched (a pair may end up with no primitives and then contributes
  // nothing).
  if (h->prim_cut > 0.0) {
    const size_t np = pairs.size();
    std::vector<double> bound(prims.size()), pmax(np, 0.0);
    std::vector<int> pair_pc(np);
    for (int pc = 0; pc < kNumPairClasses; ++pc)
      for (int32_t p : class_pairs[pc]) pair_pc[p] = pc;
    for (size_t ip = 0; ip < np; ++ip) {
      const PairRec &r = pairs[ip];
      const int lsum = kPairL[pair_pc[ip]][0] + kPairL[pair_pc[ip]][1];
      for (int k = 0; k < r.nprim; ++k) {
        const PrimRec &q = prims[r.prim_off + k];
        const double pa = std::sqrt(q.PAx * q.PAx + q.PAy * q.PAy + q.PAz * q.PAz);
        const double b = std::sqrt(kTwoPi52) * std::fabs(q.K) * std::pow(1.0 + pa + 1.0 / std::sqrt(q.p), lsum);
        bound[r.prim_off + k] = b;
        pmax[ip] = std::max(pmax[ip], b);
      }
    }
    // partners through the quartet test: pairs by Schwarz value descending,
    // running maximum of their bounds
    std::vector<int32_t> byx(np);
    for (size_t ip = 0; ip < np; ++ip) byx[ip] = (int32_t)ip;
    std::sort(byx.begin(), byx.end(), [&](int32_t a, int32_t b) { return pair_x[a] > pair_x[b]; });
    std::vector<double> xdesc(np), runmax(np);
    for (size_t k = 0; k < np; ++k) {
      xdesc[k] = pair_x[byx[k]];
      runmax[k] = std::max(k ? runmax[k - 1] : 0.0, pmax[byx[k]]);
    }
    // partners in the classes without a quartet test: the other list's pairs
    std::vector<double> class_max(kNumPairClasses, 0.0), untested(kNumPairClasses, 0.0);
    for (size_t ip = 0; ip < np; ++ip) class_max[pair_pc[ip]] = std::max(class_max[pair_pc[ip]], pmax[ip]);
    for (int c = 0; c < kNumClasses; ++c)
      if (kClasses[c].cmp == CMP_NONE) {
        untested[kClasses[c].bra] = std::max(untested[kClasses[c].bra], class_max[kClasses[c].ket]);
        untested[kClasses[c].ket] = std::max(untested[kClasses[c].ket], class_max[kClasses[c].bra]);
      }
    std::vector<PrimRec> kept;
    kept.reserve(prims.size());
    for (size_t ip = 0; ip < np; ++ip) {
      PairRec &r = pairs[ip];
      double m = untested[pair_pc[ip]];
      if (pair_x[ip] > 0.0) {
        // x_cd >= cutoff / x_ab, with a margin for the rounding of the quotient
        const double t = h->schwarz_cut / pair_x[ip] * (1.0 - 1e-12);
        const size_t n = (size_t)(std::upper_bound(xdesc.begin(), xdesc.end(), t, std::greater<double>()) - xdesc.begin());
        if (n > 0) m = std::max(m, runmax[n - 1]);
      }
      const int32_t off = (int32_t)kept.size();
      for (int k = 0; k < r.nprim; ++k)
        if (bound[r.prim_off + k] * m >= h->prim_cut) kept.push_back(prims[r.prim_off + k]);
      r.prim_off = off;
      r.nprim = (int32_t)kept.size() - off;
    }
    h->stats.prim_pairs_dropped = (int64_t)(prims.size() - kept.size());
    prims.swap(kept);
  }
  // ---- device order.  Pairs of one class sorted by (kept primitives, Schwarz
  // value descending, shell order): every class's kept list is then a run of
  // consecutive pairs per primitive count (its pre-screen keeps the largest
  // Schwarz values), and so are the kets of a segment.  The k-th primitive
  // records of the pairs of one run are consecutive as well, so that the lanes
  // of a row tile read neighbouring 64-byte records (207 G records/s against
  // 103 G for scattered ones).
  {
    std::vector<PairRec> sorted;
    std::vector<double> sorted_x;
    std::vector<PrimRec> laid;
    sorted.reserve(pairs.size());
    sorted_x.reserve(pairs.size());
    laid.reserve(prims.size());
    // (a Schwarz value that is not a number is never kept: last)
    auto key = [&](int32_t p) { return pair_x[p] == pair_x[p] ? pair_x[p] : -INFINITY; };
    for (auto &list : class_pairs) {
      std::sort(list.begin(), list.end(), [&](int32_t a, int32_t b) {
        if (pairs[a].nprim != pairs[b].nprim) return pairs[a].nprim < pairs[b].nprim;
        if (key(a) != key(b)) return key(a) > key(b);
        return a < b;
      });
      for (size_t g0 = 0, g1; g0 < list.size(); g0 = g1) {
        const int np = pairs[list[g0]].nprim;
        for (g1 = g0; g1 < list.size() && pairs[list[g1]].nprim == np;) ++g1;
        const int32_t off = (int32_t)laid.size(), n = (int32_t)(g1 - g0);
        for (int k = 0; k < np; ++k)
          for (size_t j = g0; j < g1; ++j) laid.push_back(prims[pairs[list[j]].prim_off + k]);
        for (int32_t j = 0; j < n; ++j) {
          const int32_t p = list[g0 + j];
          sorted.push_back(pairs[p]);
          // (a pair without primitives has no record: an offset in the array all the same)
          sorted.back().prim_off = np > 0 ? off + j : 0;
          sorted.back().prim_stride = n;
          sorted_x.push_back(pair_x[p]);
          list[g0 + j] = (int32_t)sorted.size() - 1;
        }
      }
    }
    pairs.swap(sorted);
    pair_x.swap(sorted_x);
    prims.swap(laid);
    PairLayout &pl = h->layout = PairLayout{};
    int64_t off = 0;
    int32_t first = 0;
    for (int pc = 0; pc < kNumPairClasses; ++pc) {
      pl.off[pc] = off;
      pl.first[pc] = first;
      pl.n[pc] = (int32_t)class_pairs[pc].size();
      const int64_t comps = (int64_t)ncart_host(kPairL[pc][0]) * ncart_host(kPairL[pc][1]);
      off += pl.n[pc] * comps;
      first += pl.n[pc];
      // workgroups of 256 pairs each per component (fewer for the largest bases)
      pl.chunks[pc] = (int32_t)std::min<int64_t>((pl.n[pc] + 255) / 256, 4096);
      pl.block[pc + 1] = pl.block[pc] + (int32_t)(pl.chunks[pc] * comps);
    }
    pl.off[kNumPairClasses] = off;
  }
  h->stats.prim_pairs = (int64_t)prims.size();

  int rc;
  if ((rc = dev_upload(h, h->pairs, pairs))) return rc;
  if ((rc = dev_upload(h, h->prims, prims))) return rc;
  const int64_t ntri = (int64_t)num_bas * (num_bas + 1) / 2;
  if ((rc = dev_alloc(h, h->dens, ntri * sizeof(double)))) return rc;
  if ((rc = dev_alloc(h, h->aux, 2 * sizeof(double)))) return rc;
  if (int e = launch_fill_zero((double *)h->aux.p, 2, h->stream))
    return fail(LIBERI_EDEVICE, std::string("zero aux: ") + hipGetErrorString((hipError_t)e));
  if ((rc = dev_alloc(h, h->fock, ntri * sizeof(double)))) return rc;
  const size_t npl = (size_t)h->layout.off[kNumPairClasses];
  const size_t nsq = (size_t)num_bas * num_bas;
  if ((rc = dev_alloc(h, h->dpair, 2 * npl * sizeof(double))) ||
      (rc = dev_alloc(h, h->jpair, 2 * npl * sizeof(double))) || (rc = dev_alloc(h, h->dsq, nsq * sizeof(double))) ||
      (rc = dev_alloc(h, h->ksq, nsq * sizeof(double))))
    return rc;

  // ---- per class: pair pre-screen (host), quartet segments (device, the
  // classes of a batch in one launch), row tiles (host).  One upload and one
  // launch a batch, one buffer for all tables: as twenty allocations a class
  // they took most of a small molecule's setup.
  struct Plan {
    int c;
    bool transposed, diag;
    std::vector<int32_t> kb, kk, gbeg;
    int64_t len0;  // the class's first segment length in the batch
  };
  std::vector<Plan> plans;
  std::vector<SegJob> jobs;
  std::vector<unsigned char> up, tab;  // uploads of the batch; the tables of all classes
  int64_t nlen = 0, nblock = 0;
  auto put = [](std::vector<unsigned char> &to, const auto &v) {
    to.resize((to.size() + 15) / 16 * 16);
    const size_t at = to.size();
    to.resize(at + v.size() * sizeof(v[0]));
    if (!v.empty()) std::memcpy(to.data() + at, v.data(), v.size() * sizeof(v[0]));
    return at;
  };
  // (pointers into the tables are offsets until they are uploaded)
  auto put_table = [&](const auto &v, auto *&p) -> int {
    const size_t before = tab.size();
    p = (std::remove_reference_t<decltype(p)>)put(tab, v);
    return charge(h, tab.size() - before);
  };
  // segments, share and tiles of a class from its segment lengths
  auto finish_class = [&](const Plan &p, const int32_t *len) -> int {
    const int c = p.c, ng = (int)p.gbeg.size();
    const ClassDef &def = kClasses[c];
    ClassState &cs_ = h->cls[c];
    int rc;
    std::vector<int64_t> sstart;
    std::vector<int32_t> sbra, sket0;
    int64_t total = 0, primq = 0;
    for (size_t i = 0; i < p.kb.size(); ++i) {
      for (int g = 0; g < ng; ++g) {
        const int64_t L = len[i * ng + g];
        if (L <= 0) continue;
        sstart.push_back(total);
        sbra.push_back(p.kb[i]);
        sket0.push_back(p.kk[p.gbeg[g]]);
        total += L;
        primq += L * (int64_t)pairs[p.kb[i]].nprim * pairs[p.kk[p.gbeg[g]]].nprim;
      }
    }
    sstart.push_back(total);
    cs_.nquart = total;
    cs_.nprimq = primq;
    if (total == 0) return LIBERI_OK;
    if (sbra.size() >= (size_t)INT32_MAX || total / kTileLens[0] + (int64_t)p.kb.size() >= (int64_t)INT32_MAX)
      return fail(LIBERI_ESIZE, std::string("class ") + def.name + ": too many segments");
    cs_.nseg = (int32_t)sbra.size();
    ClassDev &d = cs_.dev;
    if ((rc = put_table(sstart, d.seg_start)) || (rc = put_table(sbra, d.seg_bra)) ||
        (rc = put_table(sket0, d.seg_ket0)))
      return rc;
    cs_.active = true;
    d.nseg = cs_.nseg;
    d.diag = p.diag;
    // this rank's contiguous share of the class.  The reference splits each
    // class's index range into equal counts (e.g.
    // src/rhf/rot_axis/int0001.F90:100-104; LIBERI_OPT_RANK_SPLIT = 1);
    // by default the shares are equal in estimated cost instead: a quartet
    // costs its primitive quartets plus kQuartetCost for its HRR and
    // digestion, and the kept lists run from few to many primitives, so equal
    // counts leave the last ranks the most work (C60 in 8 shares, time of the
    // slowest over the mean: equal counts 1.47 to 1.50, this split 1.09 to
    // 1.11; the constant was fitted on earlier kernels, 1.08 then).
    if (h->rank_split == 1 || num_procs == 1) {
      d.q_begin = total * my_rank / num_procs;
      d.q_end = total * (my_rank + 1) / num_procs;
    } else {
      constexpr double kQuartetCost = 12.0;
      const size_t ns = sbra.size();
      std::vector<double> cum(ns + 1, 0.0), unit(ns);
      for (size_t k = 0; k < ns; ++k) {
        unit[k] = (double)pairs[sbra[k]].nprim * pairs[sket0[k]].nprim + kQuartetCost;
        cum[k + 1] = cum[k] + unit[k] * (double)(sstart[k + 1] - sstart[k]);
      }
      // first quartet at or past cost b
      auto q_at = [&](double b) -> int64_t {
        if (b <= 0.0) return 0;
        if (b >= cum[ns]) return total;
        const size_t k = (size_t)(std::upper_bound(cum.begin(), cum.end(), b) - cum.begin()) - 1;
        const int64_t q = sstart[k] + (int64_t)std::ceil((b - cum[k]) / unit[k]);
        return std::min(q, sstart[k + 1]);
      };
      d.q_begin = q_at(cum[ns] * my_rank / num_procs);
      d.q_end = my_rank + 1 == num_procs ? total : q_at(cum[ns] * (my_rank + 1) / num_procs);
    }
    // this share's primitive quartets
    {
      int64_t pq = 0;
      for (size_t k = 0; k < sbra.size(); ++k) {
        const int64_t a = std::max(sstart[k], d.q_begin), b = std::min(sstart[k + 1], d.q_end);
        if (b > a) pq += (b - a) * (int64_t)pairs[sbra[k]].nprim * pairs[sket0[k]].nprim;
      }
      primq = pq;
    }
    // (a class of at most kRowSteps workgroup steps takes one step a tile, and
    // the timed lengths where one is asked for)
    const int64_t nq = d.q_end - d.q_begin;
    cs_.small = cs_.row_ok && nq <= class_row_quartets(c) * kRowSteps;
    bool cut = true;
    // (tiles above `most` are counted, not kept)
    auto tiles_of = [&](int64_t len, const RowTile *&p, int32_t &n, size_t most = INT32_MAX) -> int {
      const std::vector<RowTile> tiles = row_tiles(c, d.q_begin, d.q_end, primq, len, cut, sstart, sbra, sket0, pairs);
      if (tiles.size() > (size_t)INT32_MAX)
        return fail(LIBERI_ESIZE, std::string("class ") + def.name + ": too many row tiles");
      n = (int32_t)tiles.size();
      return tiles.size() <= most ? put_table(tiles, p) : LIBERI_OK;
    };
    for (int k = 0; cs_.row_ok && k < kNumTileLens; ++k) {
      if (!cut) {  // no row is longer than the last length
        cs_.tiles[k] = cs_.tiles[k - 1];
        cs_.ntile[k] = cs_.ntile[k - 1];
      } else if ((rc = tiles_of(kTileLens[k], cs_.tiles[k], cs_.ntile[k]))) {
        return rc;
      }
    }
    if (cs_.small && (rc = tiles_of(class_row_quartets(c), cs_.tiles[kStepTile], cs_.ntile[kStepTile]))) return rc;
    d.row_mode = 0;
    d.threads = kRowThreads[0];
    d.transposed = p.transposed;
    {
      const PairLayout &pl = h->layout;
      const int pf = p.transposed ? def.ket : def.bra, pm = p.transposed ? def.bra : def.ket;
      d.fix_base = pl.off[pf] - pl.first[pf];
      d.mov_base = pl.off[pm] - pl.first[pm];
      d.fix_n = pl.n[pf];
      d.mov_n = pl.n[pm];
      auto pair_major = [&](int pc) {
        return pl.off[pc] - (int64_t)pl.first[pc] * ncart_host(kPairL[pc][0]) * ncart_host(kPairL[pc][1]);
      };
      d.bra_q = pair_major(def.bra);
      d.ket_q = pair_major(def.ket);
    }
    d.xswitch = h->exact_large_t ? class_rys_xmax(c) : reference_switch(c);
    h->stats.quartets[c] = d.q_end - d.q_begin;
    h->stats.prim_quartets[c] = primq;
    h->stats.total_quartets += d.q_end - d.q_begin;
    // a place in a shared launch, where the class is small
    const int sl = class_shared_launch(c, p.transposed);
    if (sl >= 0 && nq > 0) {
      int64_t groups = 0;
      if (sl < kSharedRowLaunches) {
        if (cs_.small && class_row_quartets(c) == kSharedRowThreads) {
          groups = cs_.ntile[kStepTile];
          cs_.shared_tiles = cs_.tiles[kStepTile];
        } else if (cs_.row_ok && nq <= kSharedRowThreads * kSharedRowGroups) {
          int32_t n = 0;
          if ((rc = tiles_of(kSharedRowThreads, cs_.shared_tiles, n, kSharedRowGroups))) return rc;
          groups = n;
        }
      } else {
        groups = (nq + class_round_quartets(c) - 1) / class_round_quartets(c);
      }
      if (groups > 0 && groups <= (sl < kSharedRowLaunches ? kSharedRowGroups : kSharedWaveGroups)) {
        cs_.shared = sl;
        cs_.shared_groups = (int32_t)groups;
      }
    }
    return LIBERI_OK;
  };
  auto finish_batch = [&]() -> int {
    if (plans.empty()) return LIBERI_OK;
    const size_t o_jobs = put(up, jobs), o_len = (up.size() + 15) / 16 * 16;
    std::vector<int32_t> len(nlen);
    DevBuf buf;
    if (int r = dev_alloc(h, buf, o_len + nlen * sizeof(int32_t))) return r;
    auto *base = (unsigned char *)buf.p;
    hipError_t e = hipMemcpyAsync(base, up.data(), up.size(), hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess)
      e = (hipError_t)launch_segment_lengths(base, (const SegJob *)(base + o_jobs), (int32_t)jobs.size(), nblock,
                                             h->schwarz_cut, (int32_t *)(base + o_len), h->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(len.data(), base + o_len, nlen * sizeof(int32_t), hipMemcpyDeviceToHost, h->stream);
    const hipError_t es = hipStreamSynchronize(h->stream);
    h->stats.device_bytes -= (int64_t)buf.bytes;
    dev_free(buf);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) return fail(LIBERI_EDEVICE, std::string("segment generation: ") + hipGetErrorString(e));
    for (const Plan &p : plans)
      if (int r = finish_class(p, len.data() + p.len0)) return r;
    plans.clear();
    jobs.clear();
    up.clear();
    nlen = nblock = 0;
    return LIBERI_OK;
  };
  for (int c = 0; c < kNumClasses; ++c) {
    const ClassDef &def = kClasses[c];
    ClassState &cs_ = h->cls[c];
    const auto &lb = class_pairs[def.bra], &lk = class_pairs[def.ket];
    int lmax = std::max(std::max(kPairL[def.bra][0], kPairL[def.bra][1]), std::max(kPairL[def.ket][0], kPairL[def.ket][1]));
    // the driver calls the class only if its highest shell type exists
    // (src/liberi_driver.F90:69,72,80,105); an empty pair list has no quartets
    if (lists[lmax].empty() || lb.empty() || lk.empty()) continue;
    auto maxval = [&](const std::vector<int32_t> &l) {
      double m = -INFINITY;
      for (int32_t p : l) m = std::max(m, pair_x[p]);
      return m;
    };
    const double mb = maxval(lb), mk = maxval(lk);
    const double cut = h->schwarz_cut;
    const double sb = def.ps == PS_CROSS ? cut / mk : cut / mb;
    const double sk = def.ps == PS_CROSS ? cut / mb : cut / mk;
    const bool diag = def.bra == def.ket;
    auto group_key = [&](int32_t p) { return (int64_t)pairs[p].nprim; };
    // (the lists are in device order: by primitive count, Schwarz value descending)
    auto keep = [&](const std::vector<int32_t> &l, double thr) {
      std::vector<int32_t> out;
      for (int32_t p : l)
        if (pair_x[p] >= thr) out.push_back(p);
      return out;
    };
    std::vector<int32_t> kb = keep(lb, sb);
    std::vector<int32_t> kk = diag ? kb : keep(lk, sk);
    if (kb.empty() || kk.empty()) continue;
    // Orientation of the row tiles: the fixed pair of a tile keeps its
    // exchange blocks on chip, the other pair's Coulomb block goes to F per
    // quartet.  Fix the pair whose Coulomb block is larger, among the
    // orientations whose accumulators fit in LDS.  The quartet set (and the
    // count) is the same either way: the test is on the product x_bra*x_ket.
    bool transposed = false;
    {
      const int nbra = ncart_host(kPairL[def.bra][0]) * ncart_host(kPairL[def.bra][1]);
      const int nket = ncart_host(kPairL[def.ket][0]) * ncart_host(kPairL[def.ket][1]);
      const double xsw = h->exact_large_t ? class_rys_xmax(c) : reference_switch(c);
      const int64_t l0 = class_row_lds(c, 0, h->ncol, xsw), l1 = diag ? -1 : class_row_lds(c, 1, h->ncol, xsw);
      const bool fit0 = l0 >= 0, fit1 = l1 >= 0;  // (-1: no row form, or its LDS would not fit)
      transposed = fit1 && (!fit0 || nket > nbra);
      if (h->row_orient == 1 && fit0) transposed = false;
      if (h->row_orient == 2 && fit1) transposed = true;
      cs_.row_ok = fit0 || fit1;
    }
    if (transposed) kb.swap(kk);
    // ket groups (equal group key)
    std::vector<int32_t> gbeg, gend, kgroup(kk.size());
    for (size_t j = 0; j < kk.size(); ++j) {
      if (j == 0 || group_key(kk[j]) != group_key(kk[j - 1])) {
        if (j) gend.push_back((int32_t)j);
        gbeg.push_back((int32_t)j);
      }
      kgroup[j] = (int32_t)gbeg.size() - 1;
    }
    gend.push_back((int32_t)kk.size());
    const int ng = (int)gbeg.size();
    std::vector<double> bx(kb.size()), kx(kk.size());
    std::vector<int32_t> bgroup(diag ? kb.size() : 0);
    for (size_t i = 0; i < kb.size(); ++i) {
      bx[i] = pair_x[kb[i]];
      if (diag) bgroup[i] = kgroup[i];
    }
    for (size_t j = 0; j < kk.size(); ++j) kx[j] = pair_x[kk[j]];
    const int64_t nsegc = (int64_t)kb.size() * ng;
    // the class's working memory counts against the budget, one class at a time
    const size_t work = kb.size() * (sizeof(double) + 2 * sizeof(int32_t)) + kk.size() * sizeof(double) +
                        2 * ng * sizeof(int32_t) + nsegc * sizeof(int64_t);
    if ((rc = charge(h, work))) return rc;
    h->stats.device_bytes -= (int64_t)work;
    // a batch holds at most 64 MB and what the budget leaves, or one class
    // (sixteen bytes of padding an array)
    const size_t add = kb.size() * (sizeof(double) + sizeof(int32_t)) + kk.size() * sizeof(double) +
                       2 * ng * sizeof(int32_t) + nsegc * sizeof(int32_t) + sizeof(SegJob) + 7 * 16;
    const size_t batch = up.size() + (jobs.size() * sizeof(SegJob)) + nlen * sizeof(int32_t) + add;
    const double left = h->max_device_bytes > 0.0 ? h->max_device_bytes - (double)h->stats.device_bytes : INFINITY;
    if (!plans.empty() && (batch > (size_t)64 << 20 || (double)batch > left))
      if ((rc = finish_batch())) return rc;
    SegJob j;
    j.bra_x = (int64_t)put(up, bx);
    j.bra_group = (int64_t)put(up, bgroup);
    j.ket_x = (int64_t)put(up, kx);
    j.group_begin = (int64_t)put(up, gbeg);
    j.group_end = (int64_t)put(up, gend);
    j.len0 = nlen;
    j.block0 = nblock;
    j.nbra = (int32_t)kb.size();
    j.ngroup = ng;
    j.diag = diag;
    j.cmp = def.cmp;
    jobs.push_back(j);
    plans.push_back(Plan{c, transposed, diag, std::move(kb), std::move(kk), std::move(gbeg), nlen});
    nlen += nsegc;
    nblock += (nsegc + kSegThreads - 1) / kSegThreads;
  }
  if ((rc = finish_batch())) return rc;
  if ((rc = dev_alloc_charged(h->tables, tab.size()))) return rc;
  if (!tab.empty()) HIP_TRY(hipMemcpy(h->tables.p, tab.data(), tab.size(), hipMemcpyHostToDevice));
  for (ClassState &cs_ : h->cls) {
    if (!cs_.active) continue;
    auto at = [&](auto *&p) { p = (std::remove_reference_t<decltype(p)>)((unsigned char *)h->tables.p + (size_t)p); };
    at(cs_.dev.seg_start);
    at(cs_.dev.seg_bra);
    at(cs_.dev.seg_ket0);
    for (auto &t : cs_.tiles) at(t);
    at(cs_.shared_tiles);
    use_tiles(cs_, default_tile(cs_));
  }
  if ((rc = setup_fused(h)) || (rc = setup_shared(h))) return rc;
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->initialized = true;
  return LIBERI_OK;
}

int liberi_c_setup(liberi_ctx *h, int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                   const int32_t *ang_mom, const int32_t *contr_num, const int32_t *sh_loc, const int32_t *atom_num,
                   const int32_t *atom_loc, const int32_t *start_bas, const int32_t *end_bas,
                   const double *exponents, const double *cs, const double *cp, const double *cdc, const double *cf,
                   const double *coords, const double *schwrz, int32_t my_rank, int32_t num_procs) {
  (void)start_bas;  // stored but never read by the reference's hot path either
  (void)end_bas;
  if (!h) return fail(LIBERI_EARG, "liberi_c_setup: NULL handle");
  if (!schwrz) return fail(LIBERI_EARG, "liberi_c_setup: NULL array");
  if (num_procs < 1 || my_rank < 0 || my_rank >= num_procs)
    return fail(LIBERI_EARG, "liberi_c_setup: need 0 <= my_rank < num_procs");
  std::vector<HostShell> sh;
  if (int rc0 = read_shells("liberi_c_setup", nsh, natoms, num_bas, mxgtot, ang_mom, contr_num, sh_loc, atom_num,
                            atom_loc, exponents, cs, cp, cdc, cf, coords, sh))
    return rc0;
  // a set-up handle is cleaned up first (src/interface/liberi_interface.F90:133-136);
  // so is whatever an earlier setup that failed part of the way left behind
  liberi_c_cleanup(h);
  const int rc = setup_basis(h, nsh, natoms, num_bas, mxgtot, sh, schwrz, my_rank, num_procs);
  if (rc != LIBERI_OK) {
    const std::string msg = g_last_error;
    (void)hipStreamSynchronize(h->stream);
    release_device(h);
    g_last_error = msg;
  }
  return rc;
}

// ------------------------------------------------------------------ build
// Autotuner: for every class that has both a direct and a row-tiled kernel,
// time each on this build's density (into a scratch Fock matrix, best of two
// runs each) and keep the faster.  Runs once per setup, at the first build;
// classes too small to time reliably, and every class when tuning is off, take
// the default: row tiles for the lane-per-quartet classes (whose cost is the
// atomics), direct digestion for the workgroup classes (whose occupancy the
// LDS accumulators would cut).
constexpr int64_t kTuneMinQuartets = 20000;
constexpr float kTileGain = 0.06f, kThreadsGain = 0.02f;
constexpr int kBranches = 4;  // of the batched form (one hardware queue each)
// latency of each shared launch, with few quartets in its classes (measured on
// ethane and the 3-atom C-N chain, ms)
constexpr double kSharedMs[kSharedLaunches] = {0.03, 0.06, 0.1, 0.05, 0.1, 0.08};

// Choices made so far in this process: later handles (a request loop sets up
// one per molecule) reuse them instead of timing again, but only for a class
// of about the same size -- the key is the class and its quartet count to
// within a factor of 8 -- and, for the FP32 choice, the same switch tau.
static std::mutex g_tune_mu;
static std::map<std::tuple<int, int, double>, int> g_tuned;  // (class, size, tau or -1) -> choice

// classes within a factor of 8 in quartet count share a choice
static int size_bucket(int64_t nq) {
  int b = 0;
  while (nq > 1) nq >>= 1, ++b;
  return b / 3;
}

static int tuned_choice(int c, int64_t nq, double tau) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tuned.find({c, size_bucket(nq), tau});
  return it == g_tuned.end() ? -1 : it->second;
}

static void set_tuned_choice(int c, int64_t nq, double tau, int v) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tuned[{c, size_bucket(nq), tau}] = v;
}

// Measured time of a class's launch and its primitive quartets, by class and
// size as above: later handles scale it to theirs.
static std::map<std::pair<int, int>, std::pair<float, int64_t>> g_class_ms;

static float scaled_class_ms(int c, int64_t nq, int64_t primq) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_class_ms.find({c, size_bucket(nq)});
  if (it == g_class_ms.end()) return -1.f;
  return it->second.first * (float)((double)std::max<int64_t>(primq, 1) / (double)std::max<int64_t>(it->second.second, 1));
}

static void set_class_ms(int c, int64_t nq, int64_t primq, float ms) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_class_ms[{c, size_bucket(nq)}] = {ms, primq};
}

static void forget_tuned_choices() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tuned.clear();
  g_class_ms.clear();
}

// Whether class c runs its row-tiled kernel in this build.
static bool class_row_mode(const liberi_ctx *h, int c) {
  const ClassState &cs_ = h->cls[c];
  return cs_.row_ok && cs_.dev.ntile > 0 &&
         (h->row_tiles == 2 || (h->row_tiles == 1 && cs_.variant == 1));
}

// One launch of class c (row-tiled or direct) into the scratch Fock matrix,
// timed with events on st.
static int time_class(liberi_ctx *h, const BuildArgs &ba, hipStream_t st, int c, bool row_mode, bool fp32,
                      float &ms) {
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  if (!h->tune_F.p)
    if (int rc = dev_alloc(h, h->tune_F, ntri * sizeof(double))) return rc;
  for (auto &e : h->tev)
    if (!e) HIP_TRY(hipEventCreate(&e));
  BuildArgs bt = ba;
  bt.F = (double *)h->tune_F.p;
  ClassDev cd = h->cls[c].dev;
  cd.row_mode = row_mode;
  cd.fp32 = fp32;
  HIP_TRY(hipEventRecord(h->tev[0], st));
  if (int e = launch_class(c, cd, bt, st, kCoopWorkgroups))
    return fail(LIBERI_EDEVICE, std::string("timing ") + kClasses[c].name + ": " + hipGetErrorString((hipError_t)e));
  HIP_TRY(hipEventRecord(h->tev[1], st));
  HIP_TRY(hipEventSynchronize(h->tev[1]));
  HIP_TRY(hipEventElapsedTime(&ms, h->tev[0], h->tev[1]));
  return LIBERI_OK;
}

// Whether class c runs in its shared launch in this build: unless a form, a
// tile length, the mixed form or a diagnostic is asked for, which the
// launches of one class have.
static bool class_shared(const liberi_ctx *h, int c) {
  return h->cls[c].shared >= 0 && h->autotune && h->row_tiles == 1 && h->tile_len < 0 && !(h->fp32_tau > 0.0) &&
         !h->fused && !h->class_timing && h->only_class < 0;
}

// Forms, tile lengths and times of the classes with launches of their own.
// Without `timed` (under a caller's capture, where nothing runs) those of
// earlier handles and the untimed ones.
static int choose_variants(liberi_ctx *h, const BuildArgs &ba, hipStream_t st, bool timed) {
  for (int c = 0; c < kNumClasses; ++c) {
    ClassState &cs_ = h->cls[c];
    if (!cs_.active || cs_.variant >= 0 || class_shared(h, c)) continue;
    const int64_t nq = cs_.dev.q_end - cs_.dev.q_begin;
    // untimed choice: row tiles for the lane classes, and for the group
    // classes with a wave-split form unless the class is too small to time
    const int dflt =
        (cs_.row_ok && (class_kernel_kind(c) == 0 || (class_has_split(c) && (!h->autotune || nq >= kTuneMinQuartets))))
            ? 1
            : 0;
    if (class_has_coop(c)) {
      // group class with a cooperative form (variant 3), and with a
      // wave-split row form (variant 1) where it has one: one launch of each
      // is cheap at any size, so they are timed without a size threshold
      const bool row = cs_.row_ok && cs_.dev.ntile > 0 && h->row_tiles != 0;
      cs_.variant = (dflt == 1 && h->row_tiles != 0) || h->row_tiles == 2 ? 1 : 0;
      cs_.dev.coop = 0;
      if (!h->autotune || h->row_tiles == 2 || (h->only_class >= 0 && c != h->only_class)) continue;
      if (const int prev = tuned_choice(c, nq, -3.0); prev >= 0 && (prev != 1 || row)) {
        cs_.variant = prev;
        cs_.dev.coop = prev == 3;
        continue;
      }
      if (!timed) continue;
      const int forms[3] = {0, 3, 1};  // group, cooperative, wave-split rows
      float best[3] = {1e30f, 1e30f, 1e30f};
      for (int rep = 0; rep < 6; ++rep) {
        const int k = rep % 3;
        if (forms[k] == 1 && !row) continue;
        float ms = 0.f;
        cs_.dev.coop = forms[k] == 3;
        if (int rc = time_class(h, ba, st, c, forms[k] == 1, false, ms)) return rc;
        best[k] = std::min(best[k], ms);
      }
      const int kbest = best[1] < best[0] ? (best[2] < best[1] ? 2 : 1) : (best[2] < best[0] ? 2 : 0);
      cs_.variant = forms[kbest];
      cs_.dev.coop = cs_.variant == 3;
      cs_.ms = best[kbest];
      set_tuned_choice(c, nq, -3.0, cs_.variant);
      continue;
    }
    if (!h->autotune || h->row_tiles != 1 || !cs_.row_ok || nq < kTuneMinQuartets || cs_.dev.ntile <= 0 ||
        (h->only_class >= 0 && c != h->only_class)) {
      cs_.variant = dflt;
      continue;
    }
    if (const int prev = tuned_choice(c, nq, -1.0); prev >= 0 || !timed) {
      cs_.variant = prev >= 0 ? prev : dflt;
      continue;
    }
    float best[2] = {1e30f, 1e30f};
    for (int rep = 0; rep < 4; ++rep) {
      const int v = rep & 1;
      float ms = 0.f;
      if (int rc = time_class(h, ba, st, c, v == 1, false, ms)) return rc;
      best[v] = std::min(best[v], ms);
    }
    cs_.variant = best[1] < best[0] ? 1 : 0;
    cs_.ms = std::min(best[0], best[1]);
    set_tuned_choice(c, nq, -1.0, cs_.variant);
  }
  // row-tile length of the row-tiled classes (of those of few quartets only the
  // time and the threads): shorter tiles give more
  // workgroups and more flushes of the exchange rows, longer ones fewer
  // workgroups (rows longer than a tile are split)
  for (int c = 0; c < kNumClasses; ++c) {
    ClassState &cs_ = h->cls[c];
    if (!cs_.active || cs_.tile >= 0 || class_shared(h, c)) continue;
    const int64_t nq = cs_.dev.q_end - cs_.dev.q_begin;
    cs_.tile = h->tile_len >= 0 ? h->tile_len : default_tile(cs_);
    cs_.dev.threads = kRowThreads[0];
    if (h->tile_len >= 0 || !h->autotune || !class_row_mode(h, c) || nq < kTuneMinQuartets ||
        (h->only_class >= 0 && c != h->only_class)) {
      use_tiles(cs_, cs_.tile);
      continue;
    }
    if (const int prev = tuned_choice(c, nq, -2.0); prev >= 0) {
      cs_.tile = cs_.small ? kStepTile : std::min(prev, kNumTileLens - 1);
      use_tiles(cs_, cs_.tile);
      if (tuned_choice(c, nq, -4.0) == 1) cs_.dev.threads = kRowThreads[1];
      continue;
    }
    if (!timed) {
      use_tiles(cs_, cs_.tile);
      continue;
    }
    float best[kNumTileLens + 1];
    const int k0 = cs_.small ? kStepTile : 0, k1 = cs_.small ? kStepTile : kNumTileLens - 1;
    for (int k = k0; k <= k1; ++k) best[k] = 1e30f;
    for (int rep = 0; rep < 2; ++rep)
      for (int k = k0; k <= k1; ++k) {
        if (cs_.ntile[k] <= 0) continue;
        use_tiles(cs_, k);
        float ms = 0.f;
        if (int rc = time_class(h, ba, st, c, true, false, ms)) return rc;
        best[k] = std::min(best[k], ms);
      }
    // the longest one unless a shorter is clearly faster: alone, short tiles
    // fill the tail of a class, but in a build the other classes do that, and
    // each tile costs a flush (one of 8 rank shares of C60: 4096 for every
    // class 10.6 ms, 512 12.2, the fastest of each class alone 10.7)
    cs_.tile = k1;
    for (int k = k1 - 1; k >= k0; --k)
      if (best[k] < (1.f - kTileGain) * best[cs_.tile]) cs_.tile = k;
    use_tiles(cs_, cs_.tile);
    cs_.ms = best[cs_.tile];
    // workgroup size of the lane classes, with those tiles
    if (class_kernel_kind(c) == 0) {
      cs_.dev.threads = kRowThreads[1];
      float b = 1e30f;
      for (int rep = 0; rep < 2; ++rep) {
        float ms = 0.f;
        if (int rc = time_class(h, ba, st, c, true, false, ms)) return rc;
        b = std::min(b, ms);
      }
      const bool wide = b < (1.f - kThreadsGain) * cs_.ms;
      if (wide) cs_.ms = b;
      cs_.dev.threads = kRowThreads[wide];
      set_tuned_choice(c, nq, -4.0, wide);
    }
    set_tuned_choice(c, nq, -2.0, cs_.tile);
  }
  // mixed form: FP32 stays on only in the classes where it is measured
  // faster than FP64 by at least kFp32Gain (without packed FP32 an FP32
  // instruction costs what an FP64 one does, so most classes lose by the
  // conversions); the lane-per-quartet classes have an FP32 path
  constexpr float kFp32Gain = 0.02f;
  for (int c = 0; c < kNumClasses; ++c) {
    ClassState &cs_ = h->cls[c];
    if (!cs_.active || cs_.fp32 >= 0 || class_shared(h, c)) continue;
    const int64_t nq = cs_.dev.q_end - cs_.dev.q_begin;
    // (the cooperative form, (fs|fs)'s choice, has no FP32 path either)
    if (!(h->fp32_tau > 0.0) || class_kernel_kind(c) != 0 || (cs_.dev.coop && !class_row_mode(h, c))) {
      cs_.fp32 = h->fp32_tau > 0.0 ? 0 : -1;
      continue;
    }
    if (!h->autotune || nq < kTuneMinQuartets || (h->only_class >= 0 && c != h->only_class)) {
      cs_.fp32 = 1;  // untimed: the form as asked for
      continue;
    }
    if (const int prev = tuned_choice(c, nq, h->fp32_tau); prev >= 0 || !timed) {
      cs_.fp32 = prev >= 0 ? prev : 1;
      continue;
    }
    float best[2] = {1e30f, 1e30f};
    for (int rep = 0; rep < 4; ++rep) {
      const int v = rep & 1;
      float ms = 0.f;
      if (int rc = time_class(h, ba, st, c, class_row_mode(h, c), v == 1, ms)) return rc;
      best[v] = std::min(best[v], ms);
    }
    cs_.fp32 = best[1] < (1.f - kFp32Gain) * best[0] ? 1 : 0;
    set_tuned_choice(c, nq, h->fp32_tau, cs_.fp32);
  }
  if (!timed) return LIBERI_OK;
  // the time of every class not timed above, which spreads the classes over
  // the branches: from an earlier handle, or the second of two launches
  // (the first one of a kernel in the process loads its code, up to
  // milliseconds)
  for (int c = 0; c < kNumClasses; ++c) {
    ClassState &cs_ = h->cls[c];
    if (!cs_.active || class_shared(h, c) || (h->only_class >= 0 && c != h->only_class)) continue;
    const int64_t nq = cs_.dev.q_end - cs_.dev.q_begin, primq = h->stats.prim_quartets[c];
    if (cs_.ms < 0.f && (cs_.ms = scaled_class_ms(c, nq, primq)) >= 0.f) continue;
    for (int rep = 0; cs_.ms < 0.f && rep < 2; ++rep) {
      float ms = 0.f;
      if (int rc = time_class(h, ba, st, c, class_row_mode(h, c), cs_.fp32 == 1, ms)) return rc;
      if (rep == 1) cs_.ms = ms;
    }
    set_class_ms(c, nq, primq, cs_.ms);
  }
  return LIBERI_OK;
}

// max |D| of the build into aux[0] and a zero FP32 quartet count into aux[1]
// (the mixed form's switch reads them)
static int enqueue_dmax(liberi_ctx *h, const double *dD, hipStream_t st) {
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  int e = launch_fill_zero((double *)h->aux.p, 2, st);
  if (e == hipSuccess) e = launch_abs_max(dD, ntri, (double *)h->aux.p, st);
  if (e != hipSuccess) return fail(LIBERI_EDEVICE, std::string("max |D|: ") + hipGetErrorString((hipError_t)e));
  return LIBERI_OK;
}

static BuildWork build_work(const BuildArgs &ba) {
  return BuildWork{const_cast<double *>(ba.Dp), const_cast<double *>(ba.Dq), const_cast<double *>(ba.Dsq)};
}

// Zero F (and find max |D| for the mixed form), then every class's kernel.
// With ns > 1, under capture on st, the classes are spread over ns branches of
// the graph, longest first onto the least-loaded branch: a launch is captured
// behind the last one of its branch.  (One stream captures them all; a stream
// per branch took 0.5 ms to create and destroy, most of a request's teardown.)
// `spins` builds of one basis (their arguments at bas, each its own
// workspace) go side by side: the two Fock matrices of an unrestricted build.
static int enqueue_build(liberi_ctx *h, const BuildArgs *bas, int spins, const double *dD, hipStream_t st, int ns) {
  // fock = 0 (src/liberi_driver.F90:64)
  for (int s = 0; s < spins; ++s)
    if (int e = launch_build_begin(bas[s], h->layout, build_work(bas[s]), st))
      return fail(LIBERI_EDEVICE, std::string("start of the build: ") + hipGetErrorString((hipError_t)e));
  if (h->fp32_tau > 0.0)
    if (int rc = enqueue_dmax(h, dD, st)) return rc;
  // (nothing to time under a caller's capture)
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIP_TRY(hipStreamIsCapturing(st, &cap));
  const bool timing = h->class_timing && cap == hipStreamCaptureStatusNone;
  // the fused group launch, where on: its classes leave the per-class launches
  const bool fused = h->fused && h->fused_n > 0 && !h->class_timing && h->only_class < 0;
  auto ran = [&](int c, int variant, int64_t tile, bool fp32) {
    ClassState &cs_ = h->cls[c];
    cs_.ran = variant;
    cs_.ran_tile = (int32_t)tile;
    cs_.ran_fp32 = fp32;
  };
  // launches of the build, by cost (ms): a class (its measured time, else the
  // proxy), or kNumClasses + k for shared launch k
  auto cost = [&](int c) { return h->cls[c].ms >= 0.f ? (double)h->cls[c].ms : class_cost_proxy(h, c); };
  std::vector<std::pair<double, int>> order;
  double shared_cost[kSharedLaunches] = {};
  double fused_cost = 0.0;
  for (int c = 0; c < kNumClasses; ++c)
    if (h->cls[c].active && (h->only_class < 0 || c == h->only_class)) {
      const ClassState &cs_ = h->cls[c];
      if (fused && class_fused_nq(c) > 0) {
        ran(c, 4, 0, false);
      } else if (class_shared(h, c)) {
        shared_cost[cs_.shared] += class_cost_proxy(h, c);
        if (cs_.shared < kSharedRowLaunches)
          ran(c, 1 + cs_.dev.transposed, kSharedRowThreads, false);
        else
          ran(c, cs_.shared > kSharedGroupLaunch ? 3 : 0, 0, false);
      } else {
        order.push_back({cost(c), c});
        const bool row = class_row_mode(h, c), coop = !row && (cs_.dev.coop || class_kernel_kind(c) == 2);
        ran(c, row ? 1 + cs_.dev.transposed : coop ? 3 : 0, row ? tile_length(c, cs_.tile) : 0,
            h->fp32_tau > 0.0 && cs_.fp32 == 1 && !coop);
      }
    }
  for (int k = 0; k < kSharedLaunches; ++k)
    if (shared_cost[k] > 0.0) order.push_back({kSharedMs[k] + shared_cost[k], kNumClasses + k});
  std::vector<double> load(ns, 0.0);
  if (ns > 1) std::sort(order.begin(), order.end(), std::greater<>());
  // captured nodes the next launch on st depends on, and the last of each branch
  using Nodes = std::vector<hipGraphNode_t>;
  auto captured = [&](Nodes &v) -> hipError_t {
    hipStreamCaptureStatus cap;
    const hipGraphNode_t *deps = nullptr;
    size_t n = 0;
    const hipError_t e = hipStreamGetCaptureInfo_v2(st, &cap, nullptr, nullptr, &deps, &n);
    if (e == hipSuccess) v.assign(deps, deps + n);
    return e;
  };
  auto depend_on = [&](Nodes &v) -> hipError_t {
    return hipStreamUpdateCaptureDependencies(st, v.data(), v.size(), hipStreamSetCaptureDependencies);
  };
  std::vector<Nodes> branch(ns);
  if (ns > 1) {
    HIP_TRY(captured(branch[0]));
    for (int k = 1; k < ns; ++k) branch[k] = branch[0];
  }
  if (fused) {
    // one persistent launch for the fused classes, first onto the least-loaded
    // stream
    for (int c = 0; c < kNumClasses; ++c)
      if (h->cls[c].active && class_fused_nq(c) > 0) fused_cost += cost(c);
    int k = 0;
    if (ns > 1) {
      k = ns > 1 ? 1 : 0;
      load[k] += fused_cost;
    }
    if (ns > 1) HIP_TRY(depend_on(branch[k]));
    int e = launch_fill_zero((double *)h->fused_head.p, 1, st);
    if (e == hipSuccess)
      e = launch_group_fused((const ClassDev *)h->fused_cds.p, bas[0], (const FusedItem *)h->fused_items.p, h->fused_n,
                             (unsigned long long *)h->fused_head.p, h->fused_nwg, st);
    if (e != hipSuccess)
      return fail(LIBERI_EDEVICE, std::string("fused group launch: ") + hipGetErrorString((hipError_t)e));
    if (ns > 1) HIP_TRY(captured(branch[k]));
  }
  for (const auto &[ms, c] : order)
    for (int s = 0; s < spins; ++s) {
      const BuildArgs &ba = bas[s];
      const int k = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      load[k] += ms;
      if (ns > 1) HIP_TRY(depend_on(branch[k]));
      if (c >= kNumClasses) {
        if (int e = launch_shared(c - kNumClasses, h->shared[c - kNumClasses], (const ClassDev *)h->shared_cds.p, ba, st))
          return fail(LIBERI_EDEVICE, std::string("shared launch: ") + hipGetErrorString((hipError_t)e));
      } else {
        if (timing) {
          if (!h->cev0[c]) HIP_TRY(hipEventCreate(&h->cev0[c]));
          if (!h->cev1[c]) HIP_TRY(hipEventCreate(&h->cev1[c]));
          HIP_TRY(hipEventRecord(h->cev0[c], st));
        }
        ClassDev cd = h->cls[c].dev;
        cd.row_mode = class_row_mode(h, c);
        cd.fp32 = h->cls[c].fp32 == 1;
        int e = launch_class(c, cd, ba, st, kCoopWorkgroups);
        if (e != hipSuccess)
          return fail(LIBERI_EDEVICE,
                      std::string("launch ") + kClasses[c].name + ": " + hipGetErrorString((hipError_t)e));
        if (timing) HIP_TRY(hipEventRecord(h->cev1[c], st));
      }
      if (ns > 1) HIP_TRY(captured(branch[k]));
    }
  if (ns > 1) {
    Nodes all;
    for (const Nodes &v : branch)
      for (hipGraphNode_t n : v)
        if (std::find(all.begin(), all.end(), n) == all.end()) all.push_back(n);
    HIP_TRY(depend_on(all));
  }
  for (int s = 0; s < spins; ++s)
    if (int e = launch_build_end(bas[s], h->layout, st))
      return fail(LIBERI_EDEVICE, std::string("end of the build: ") + hipGetErrorString((hipError_t)e));
  return LIBERI_OK;
}

// RHF: DK = D, k_scale = 1.  A UHF spin component: D = Da + Db, DK = that
// spin's density, k_scale = 2 (F_s = J[Da+Db] - K[Ds]).
static BuildArgs build_args(liberi_ctx *h, const double *dD, const double *dK, double *dF, double k_scale) {
  BuildArgs ba;
  ba.pairs = (const PairRec *)h->pairs.p;
  ba.prims = (const PrimRec *)h->prims.p;
  ba.D = dD;
  ba.DK = dK;
  ba.k_scale = k_scale;
  const int64_t npl = h->layout.off[kNumPairClasses];
  ba.Dp = (const double *)h->dpair.p;
  ba.Dq = ba.Dp + npl;
  ba.Dsq = (const double *)h->dsq.p;
  ba.Jp = (double *)h->jpair.p;
  ba.Jq = ba.Jp + npl;
  ba.Ksq = (double *)h->ksq.p;
  ba.F = dF;
  ba.value_cut = h->value_cut;
  ba.nbf = h->num_bas;
  ba.fp32_tau = h->fp32_tau;
  ba.dmax = (const double *)h->aux.p;
  ba.fp32_count = (uint64_t *)h->aux.p + 1;
  for (int l = 0; l < 4; ++l) {
    ba.col_bf[l] = (const int32_t *)h->col_bf[l].p;
    ba.ncol[l] = h->ncol[l];
  }
  return ba;
}

// doubles of a build's workspace beside the handle's own, and its arrays in `w`
static size_t work_doubles(const liberi_ctx *h) {
  return 4 * (size_t)h->layout.off[kNumPairClasses] + 2 * (size_t)h->num_bas * h->num_bas;
}
static void use_work(const liberi_ctx *h, BuildArgs &ba, double *w) {
  const size_t npl = (size_t)h->layout.off[kNumPairClasses], nsq = (size_t)h->num_bas * h->num_bas;
  ba.Dp = w;
  ba.Dq = w + npl;
  ba.Jp = w + 2 * npl;
  ba.Jq = w + 3 * npl;
  ba.Dsq = w + 4 * npl;
  ba.Ksq = w + 4 * npl + nsq;
}

// The workspace of a build into ba.F under a caller's capture.
static int use_captured_work(liberi_ctx *h, BuildArgs &ba) {
  for (const auto &[F, buf] : h->captured)
    if (F == ba.F) return use_work(h, ba, (double *)buf.p), LIBERI_OK;
  DevBuf buf;
  // (an allocation is no work of the stream's)
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
  const int rc = dev_alloc(h, buf, work_doubles(h) * sizeof(double));
  HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
  if (rc) return rc;
  h->captured.push_back({ba.F, buf});
  use_work(h, ba, (double *)buf.p);
  return LIBERI_OK;
}

// whether the next build has to choose forms, tile lengths or times first
static bool choices_open(const liberi_ctx *h) {
  for (int k = 0; k < kNumClasses; ++k) {
    const ClassState &c = h->cls[k];
    if (!c.active || class_shared(h, k)) continue;
    const bool runs = h->only_class < 0 || k == h->only_class;
    if (c.variant < 0 || c.tile < 0 || (c.ms < 0.f && runs) || (h->fp32_tau > 0.0 && c.fp32 < 0)) return true;
  }
  return false;
}

// The build of bas[0 .. spins) as branches of a graph, captured on the handle's stream.
static int capture_build(liberi_ctx *h, const BuildArgs *bas, int spins, hipGraph_t *graph, hipGraphExec_t *exec) {
  HIP_TRY(hipStreamSynchronize(h->stream));
  HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_build(h, bas, spins, bas[0].D, h->stream, kBranches);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(h->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(LIBERI_EDEVICE, std::string("graph capture: ") + hipGetErrorString(e));
  *graph = g;
  HIP_TRY(hipGraphInstantiate(exec, g, nullptr, nullptr, 0));
  return LIBERI_OK;
}

static int build_on_device(liberi_ctx *h, const double *dD, double *dF, hipStream_t st, const double *dK = nullptr,
                           double k_scale = 1.0) {
  BuildArgs ba = build_args(h, dD, dK ? dK : dD, dF, k_scale);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIP_TRY(hipStreamIsCapturing(st, &cap));
  const bool runs = cap == hipStreamCaptureStatusNone;
  if (runs && h->built) HIP_TRY(hipStreamWaitEvent(st, h->ev1, 0));
  // (the caller may replay what is captured here beside other builds)
  if (!runs)
    if (int rc = use_captured_work(h, ba)) return rc;
  // the autotuner's timed launches see this build's max |D| (mixed form)
  if (h->fp32_tau > 0.0)
    if (int rc = enqueue_dmax(h, dD, st)) return rc;
  // (they also run before any build: Dp and Dsq from this build's density)
  // (choices made under a caller's capture are untimed, and for that build only)
  struct Choices {
    liberi_ctx *h;
    std::vector<ClassState> cls;
    ~Choices() {
      for (size_t c = 0; c < cls.size(); ++c) {
        const ClassState &now = h->cls[c];
        cls[c].ran = now.ran, cls[c].ran_tile = now.ran_tile, cls[c].ran_fp32 = now.ran_fp32;
        h->cls[c] = cls[c];
      }
    }
  } choices{h, {}};
  if (choices_open(h)) {
    if (!runs) {
      choices.cls.assign(h->cls, h->cls + kNumClasses);
    } else if (int e = launch_build_begin(ba, h->layout, build_work(ba), st)) {
      return fail(LIBERI_EDEVICE, std::string("start of the build: ") + hipGetErrorString((hipError_t)e));
    }
    if (int rc = choose_variants(h, ba, st, runs)) return rc;
  }
  // the batched form: capture once (per D, F), replay afterwards; under a
  // caller's capture, its branches straight into the caller's graph.  Per-class
  // timing and single-class diagnostics run eagerly on st.
  const bool batched = h->use_graph && !h->class_timing && h->only_class < 0 && ba.DK == dD && k_scale == 1.0;
  const bool graph = batched && runs;
  // (a graph of other arrays may still run: it goes after the launch of the new one)
  hipGraph_t no_graph = nullptr;
  hipGraphExec_t no_exec = nullptr;
  const bool recapture = graph && (!h->gexec || h->g_dD != dD || h->g_dF != dF);
  OldGraph old(h, recapture ? h->graph : no_graph, recapture ? h->gexec : no_exec);
  if (recapture) {
    if (int rc = capture_build(h, &ba, 1, &h->graph, &h->gexec)) return rc;
    h->g_dD = dD;
    h->g_dF = dF;
  }
  if (runs) HIP_TRY(hipEventRecord(h->ev0, st));
  if (graph) {
    HIP_TRY(hipGraphLaunch(h->gexec, st));
  } else if (int rc = enqueue_build(h, &ba, 1, dD, st, batched ? kBranches : 1)) {
    return rc;
  }
  old.end();
  if (runs) HIP_TRY(end_build(h, st));
  h->build_pending = true;
  h->fp32_pending = h->fp32_tau > 0.0;
  if (!h->fp32_pending) h->stats.fp32_quartets = 0;
  h->timing_pending = h->class_timing && !graph && runs;
  if (!h->timing_pending)
    for (double &v : h->stats.class_ms) v = 0.0;
  return LIBERI_OK;
}

int liberi_c_fock_build(liberi_ctx *h, const double *density, double *fock, int64_t n) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_fock_build: NULL handle");
  if (!h->initialized)
    return fail(LIBERI_ESTATE, "liberi_fock_build called before liberi_setup");  // liberi_interface.F90:219-222
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  if (n != ntri)
    return fail(LIBERI_ESIZE, "liberi_c_fock_build: n=" + std::to_string(n) + ", expected " + std::to_string(ntri));
  if (!density || !fock) return fail(LIBERI_EARG, "liberi_c_fock_build: NULL array");
  HIP_TRY(hipMemcpyAsync(h->dens.p, density, ntri * sizeof(double), hipMemcpyHostToDevice, h->stream));
  int rc = build_on_device(h, (const double *)h->dens.p, (double *)h->fock.p, h->stream);
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(fock, h->fock.p, ntri * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  collect_timing(h);
  return LIBERI_OK;
}

int liberi_c_fock_build_device(liberi_ctx *h, const double *dD, double *dF, int64_t n, void *stream) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_fock_build_device: NULL handle");
  if (!h->initialized) return fail(LIBERI_ESTATE, "liberi_fock_build called before liberi_setup");
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  if (n != ntri)
    return fail(LIBERI_ESIZE, "liberi_c_fock_build_device: n=" + std::to_string(n) + ", expected " + std::to_string(ntri));
  if (!dD || !dF) return fail(LIBERI_EARG, "liberi_c_fock_build_device: NULL array");
  return build_on_device(h, dD, dF, stream ? (hipStream_t)stream : h->stream);
}

// ------------------------------------------------------------------- UHF
// Both spins' builds side by side in one graph, from the second call on the
// same four arrays on (one after the other on one stream, the 17-atom
// cluster's classes leave the chip idle most of the time: 973 -> 832 us).  The
// second build has a workspace of its own.  Returns 1 when the builds have to
// run one after the other, 0 when done, else an error.
static int build_uhf_graph(liberi_ctx *h, const double *dt, const double *dDa, const double *dDb, double *dFa,
                           double *dFb, hipStream_t st, int *rc) {
  *rc = LIBERI_OK;
  const void *arrays[4] = {dDa, dDb, dFa, dFb};
  const bool again = std::equal(arrays, arrays + 4, h->u_arrays);
  std::copy(arrays, arrays + 4, h->u_arrays);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (!again || h->uhf_refused || !h->use_graph || h->class_timing || h->only_class >= 0 || h->fused || h->fp32_tau > 0.0 ||
      choices_open(h) || hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
    return 1;
  hipGraph_t no_graph = nullptr;
  hipGraphExec_t no_exec = nullptr;
  const bool recapture = !h->uexec || !std::equal(arrays, arrays + 4, h->ug_arrays);
  OldGraph old(h, recapture ? h->ugraph : no_graph, recapture ? h->uexec : no_exec);
  if (recapture) {
    if (!h->uhf_work.p) {
      const std::string msg = g_last_error;
      if (dev_alloc(h, h->uhf_work, work_doubles(h) * sizeof(double)) != LIBERI_OK) {
        h->uhf_refused = true;
        g_last_error = msg;
        return 1;
      }
    }
    BuildArgs bas[2] = {build_args(h, dt, dDa, dFa, 2.0), build_args(h, dt, dDb, dFb, 2.0)};
    use_work(h, bas[1], (double *)h->uhf_work.p);
    if ((*rc = capture_build(h, bas, 2, &h->ugraph, &h->uexec))) return 0;
    std::copy(arrays, arrays + 4, h->ug_arrays);
  }
  hipError_t e = h->built ? hipStreamWaitEvent(st, h->ev1, 0) : hipSuccess;
  if (e == hipSuccess) e = (hipError_t)launch_add(dDa, dDb, const_cast<double *>(dt), (int64_t)h->num_bas * (h->num_bas + 1) / 2, st);
  if (e == hipSuccess) e = hipEventRecord(h->ev0, st);
  if (e == hipSuccess) e = hipGraphLaunch(h->uexec, st);
  old.end();
  if (e == hipSuccess) e = end_build(h, st);
  if (e != hipSuccess) {
    *rc = fail(LIBERI_EDEVICE, std::string("UHF build: ") + hipGetErrorString(e));
    return 0;
  }
  h->build_pending = true;
  h->fp32_pending = h->timing_pending = false;
  h->stats.fp32_quartets = 0;
  for (double &v : h->stats.class_ms) v = 0.0;
  return 0;
}

int liberi_c_fock_build_uhf_device(liberi_ctx *h, const double *dDa, const double *dDb, double *dFa, double *dFb,
                                   int64_t n, void *stream) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_fock_build_uhf_device: NULL handle");
  if (!h->initialized) return fail(LIBERI_ESTATE, "liberi_fock_build called before liberi_setup");
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  if (n != ntri)
    return fail(LIBERI_ESIZE, "liberi_c_fock_build_uhf_device: n=" + std::to_string(n) + ", expected " + std::to_string(ntri));
  if (!dDa || !dDb || !dFa || !dFb) return fail(LIBERI_EARG, "liberi_c_fock_build_uhf_device: NULL array");
  hipStream_t st = stream ? (hipStream_t)stream : h->stream;
  if (!h->dens_t.p)
    if (int rc = dev_alloc(h, h->dens_t, ntri * sizeof(double))) return rc;
  double *dt = (double *)h->dens_t.p;
  int rcu = LIBERI_OK;
  if (!build_uhf_graph(h, dt, dDa, dDb, dFa, dFb, st, &rcu)) return rcu;
  // Da + Db is written where a build on another stream may still read it
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIP_TRY(hipStreamIsCapturing(st, &cap));
  if (cap == hipStreamCaptureStatusNone && h->built) HIP_TRY(hipStreamWaitEvent(st, h->ev1, 0));
  if (int e = launch_add(dDa, dDb, dt, ntri, st))
    return fail(LIBERI_EDEVICE, std::string("Da + Db: ") + hipGetErrorString((hipError_t)e));
  if (int rc = build_on_device(h, dt, dFa, st, dDa, 2.0)) return rc;
  return build_on_device(h, dt, dFb, st, dDb, 2.0);
}

int liberi_c_fock_build_uhf(liberi_ctx *h, const double *Da, const double *Db, double *Fa, double *Fb, int64_t n) {
  if (!h) return fail(LIBERI_EARG, "liberi_c_fock_build_uhf: NULL handle");
  if (!h->initialized) return fail(LIBERI_ESTATE, "liberi_fock_build called before liberi_setup");
  const int64_t ntri = (int64_t)h->num_bas * (h->num_bas + 1) / 2;
  if (n != ntri)
    return fail(LIBERI_ESIZE, "liberi_c_fock_build_uhf: n=" + std::to_string(n) + ", expected " + std::to_string(ntri));
  if (!Da || !Db || !Fa || !Fb) return fail(LIBERI_EARG, "liberi_c_fock_build_uhf: NULL array");
  if (!h->dens_b.p)
    if (int rc = dev_alloc(h, h->dens_b, ntri * sizeof(double))) return rc;
  if (!h->fock_b.p)
    if (int rc = dev_alloc(h, h->fock_b, ntri * sizeof(double))) return rc;
  const size_t bytes = ntri * sizeof(double);
  HIP_TRY(hipMemcpyAsync(h->dens.p, Da, bytes, hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(h->dens_b.p, Db, bytes, hipMemcpyHostToDevice, h->stream));
  if (int rc = liberi_c_fock_build_uhf_device(h, (const double *)h->dens.p, (const double *)h->dens_b.p,
                                              (double *)h->fock.p, (double *)h->fock_b.p, n, h->stream))
    return rc;
  HIP_TRY(hipMemcpyAsync(Fa, h->fock.p, bytes, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipMemcpyAsync(Fb, h->fock_b.p, bytes, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  collect_timing(h);
  return LIBERI_OK;
}

// ------------------------------------------- GAMESS direct-link entry points
static liberi_ctx *g_handle = nullptr;  // gms_liberi_wrapper.F90:23-25 (module `save` handle)
static int64_t g_matrix_size = 0;

int liberi_c_init(int32_t natoms, int32_t num_bas, int32_t nsh, int32_t mxgtot, const int32_t *ang_mom,
                  const int32_t *contr_num, const int32_t *sh_loc, const int32_t *atom_num, const int32_t *atom_loc,
                  const int32_t *start_bas, const int32_t *end_bas, const double *exponents, const double *cs,
                  const double *cp, const double *cd, const double *cf, const double *coords, const double *schwrz,
                  int32_t my_rank, int32_t num_procs) {
  if (g_handle) liberi_c_destroy(&g_handle);  // gms_liberi_wrapper.F90:80-83
  int rc = liberi_c_create(&g_handle);
  if (rc) return rc;
  rc = liberi_c_setup(g_handle, nsh, natoms, num_bas, mxgtot, ang_mom, contr_num, sh_loc, atom_num, atom_loc,
                      start_bas, end_bas, exponents, cs, cp, cd, cf, coords, schwrz, my_rank, num_procs);
  if (rc) {
    std::string msg = g_last_error;
    liberi_c_destroy(&g_handle);
    return fail(rc, msg);
  }
  g_matrix_size = (int64_t)num_bas * (num_bas + 1) / 2;
  return LIBERI_OK;
}

int liberi_c_fock(const double *density, double *fock, int64_t n) {
  if (!g_handle) return fail(LIBERI_ESTATE, "liberi_fock called before liberi_init");  // :117-120
  if (n != g_matrix_size)
    return fail(LIBERI_ESIZE, "matrix size mismatch in liberi_fock: expected " + std::to_string(g_matrix_size) +
                                  ", got " + std::to_string(n));  // :122-127
  return liberi_c_fock_build(g_handle, density, fock, n);
}

int liberi_c_finalize(void) {
  if (g_handle) liberi_c_destroy(&g_handle);
  g_matrix_size = 0;
  return LIBERI_OK;
}

// ------------------------------------------------------ Schwarz integrals
int liberi_c_schwarz(int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot, const int32_t *ang_mom,
                     const int32_t *contr_num, const int32_t *sh_loc, const int32_t *atom_num,
                     const int32_t *atom_loc, const double *exponents, const double *cs, const double *cp,
                     const double *cd, const double *cf, const double *coords, double *schwrz_int) {
  if (!schwrz_int) return fail(LIBERI_EARG, "liberi_c_schwarz: NULL output");
  SchwarzStage s;
  if (int rc = schwarz_stage("liberi_c_schwarz", nsh, natoms, num_bas, mxgtot, ang_mom, contr_num, sh_loc,
                             atom_num, atom_loc, exponents, cs, cp, cd, cf, coords, s))
    return rc;
  if (int rc = schwarz_check_device("liberi_c_schwarz")) return rc;
  void *buf = nullptr;
  hipStream_t st = nullptr;
  std::vector<unsigned char> host;
  std::vector<double> out(s.pairs.size());
  hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc(&buf, s.bytes);
  if (e == hipSuccess) e = (hipError_t)schwarz_enqueue(s, (unsigned char *)buf, host, st);
  if (e == hipSuccess)
    e = hipMemcpyAsync(out.data(), (unsigned char *)buf + s.o_out, out.size() * sizeof(double), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (st) (void)hipStreamDestroy(st);
  if (buf) (void)hipFree(buf);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(e == hipErrorOutOfMemory ? LIBERI_ENOMEM : LIBERI_EDEVICE,
                std::string("liberi_c_schwarz: ") + hipGetErrorString(e));
  }
  schwarz_scatter(s, out.data(), schwrz_int);
  return LIBERI_OK;
}

}  // extern "C"

// Host staging shared by the two Schwarz entry points (liberi_c_schwarz here,
// liberi_c_schwarz_noalloc in noalloc.hip).
namespace liberi {

int schwarz_stage(const char *who, int32_t nsh, int32_t natoms, int32_t num_bas, int32_t mxgtot,
                  const int32_t *ang_mom, const int32_t *contr_num, const int32_t *sh_loc, const int32_t *atom_num,
                  const int32_t *atom_loc, const double *exponents, const double *cs, const double *cp,
                  const double *cd, const double *cf, const double *coords, SchwarzStage &s) {
  std::vector<HostShell> sh;
  if (int rc = read_shells(who, nsh, natoms, num_bas, mxgtot, ang_mom, contr_num, sh_loc, atom_num, atom_loc,
                           exponents, cs, cp, cd, cf, coords, sh))
    return rc;
  s = SchwarzStage{};
  s.shells.resize(nsh);
  std::vector<double> coef;
  for (int i = 0; i < nsh; ++i) {
    s.shells[i] = SchwarzShell{sh[i].c[0], sh[i].c[1], sh[i].c[2], (int32_t)s.ew.size(), sh[i].k};
    s.ew.insert(s.ew.end(), sh[i].e, sh[i].e + sh[i].k);
    coef.insert(coef.end(), sh[i].w, sh[i].w + sh[i].k);
  }
  s.ew.insert(s.ew.end(), coef.begin(), coef.end());
  // every shell pair i >= j, A = the shell of higher angular momentum, grouped by (la, lb)
  const size_t np = (size_t)nsh * (nsh + 1) / 2;
  size_t count[17] = {};
  int64_t nprims = 0;
  for (int i = 0; i < nsh; ++i)
    for (int j = 0; j <= i; ++j) {
      ++count[std::max(sh[i].l, sh[j].l) * 4 + std::min(sh[i].l, sh[j].l) + 1];
      nprims += (int64_t)sh[i].k * sh[j].k;
    }
  if (nprims > (int64_t)INT32_MAX || np > (size_t)INT32_MAX)
    return fail(LIBERI_EARG, std::string(who) + ": basis too large for 32-bit pair indices");
  for (int k = 0; k < 16; ++k) count[k + 1] += count[k];
  std::copy(count, count + 17, s.off);
  s.pairs.resize(np);
  s.where.resize(np);
  s.nprims = nprims;
  int64_t at = 0, prim = 0;
  for (int i = 0; i < nsh; ++i)
    for (int j = 0; j <= i; ++j, ++at) {
      const int sA = sh[i].l >= sh[j].l ? i : j, sB = sA == i ? j : i, g = sh[sA].l * 4 + sh[sB].l;
      const int32_t n = sh[sA].k * sh[sB].k;
      s.longest[g] = std::max(s.longest[g], n);
      s.where[count[g]] = at;
      s.pairs[count[g]++] = SchwarzPair{sA, sB, (int32_t)prim, n};
      prim += n;
    }
  auto align256 = [](size_t n) { return (n + 255) / 256 * 256; };
  s.o_shells = np * sizeof(SchwarzPair);
  s.o_ew = s.o_shells + nsh * sizeof(SchwarzShell);
  s.upload = s.o_ew + s.ew.size() * sizeof(double);
  s.o_prims = align256(s.upload);
  s.o_out = s.o_prims + align256((size_t)nprims * sizeof(PrimRec));
  s.bytes = s.o_out + np * sizeof(double);
  return LIBERI_OK;
}

int schwarz_check_device(const char *who) {
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
    return fail(LIBERI_EDEVICE, std::string(who) + ": no HIP device visible");
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(LIBERI_EDEVICE, std::string(who) + ": device is " + prop.gcnArchName +
                                    ", this library is built for gfx950 (MI355X)");
  return LIBERI_OK;
}

int schwarz_enqueue(const SchwarzStage &s, unsigned char *buf, std::vector<unsigned char> &host, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  host.resize(s.upload);
  std::memcpy(host.data(), s.pairs.data(), s.pairs.size() * sizeof(SchwarzPair));
  std::memcpy(host.data() + s.o_shells, s.shells.data(), s.shells.size() * sizeof(SchwarzShell));
  std::memcpy(host.data() + s.o_ew, s.ew.data(), s.ew.size() * sizeof(double));
  const auto *pairs = (const SchwarzPair *)buf;
  const auto *shells = (const SchwarzShell *)(buf + s.o_shells);
  auto *prims = (PrimRec *)(buf + s.o_prims);
  auto *out = (double *)(buf + s.o_out);
  hipError_t e = hipMemcpyAsync(buf, host.data(), s.upload, hipMemcpyHostToDevice, st);
  if (e == hipSuccess)
    e = (hipError_t)launch_schwarz_records(pairs, (int32_t)s.pairs.size(), shells, (const double *)(buf + s.o_ew),
                                           (int32_t)(s.ew.size() / 2), prims, st);
  for (int k = 0; k < 16 && e == hipSuccess; ++k) {
    const int32_t n = (int32_t)(s.off[k + 1] - s.off[k]);
    if (n > 0)
      e = (hipError_t)launch_schwarz(k / 4, k % 4, pairs + s.off[k], shells, prims, n, s.longest[k], out + s.off[k], st);
  }
  return (int)e;
}

void schwarz_scatter(const SchwarzStage &s, const double *out, double *schwrz_int) {
  for (size_t k = 0; k < s.pairs.size(); ++k) schwrz_int[s.where[k]] = out[k];
}

int set_last_error(int code, const std::string &msg) { return fail(code, msg); }

}  // namespace liberi
