// The HIP calls that libliberi_hip.so makes, on the host: loaded before the
// library (RTLD_GLOBAL), this takes the runtime's place, so that what the host
// code allocates, launches, orders and frees can be seen without a GPU.
// Device memory is host memory.  Kernels do not run, but the one that the
// setup needs the results of (segment lengths).  Work on a stream is "in
// flight" until something waits for it; every stream, event and graph carries
// the work it comes after, so that a missing wait shows.
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "../gms_liberi_amd/csrc/liberi_internal.hpp"

using namespace liberi;

namespace {

using Clock = std::map<int, long>;  // stream -> work item it comes after

struct Stream {
  int id;
  Clock clock;
  bool capturing = false;
  std::string last;  // kernel launched last
  std::set<size_t> deps;
};
struct Event {
  Clock clock;
  bool recorded = false, captured = false;
  std::string last;
};
struct Exec {
  int id;
  Clock after;  // its last launch
};

std::map<int, long> g_done;
std::set<Stream *> g_streams;
std::map<void *, size_t> g_mem;
size_t g_bytes = 0, g_peak = 0, g_fail = 0;
hipError_t g_last = hipSuccess;
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
int g_next = 1;
size_t g_node = 0;
std::string g_log;
hipGraphNode_t g_deps[64];

void log(const char *fmt, ...) {
  char b[8192];
  va_list a;
  va_start(a, fmt);
  vsnprintf(b, sizeof b, fmt, a);
  va_end(a);
  g_log += b;
  g_log += '\n';
}
hipError_t err(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
void done(const Clock &c) {
  for (auto &[s, n] : c) g_done[s] = std::max(g_done[s], n);
}
bool in_flight(const Clock &c) {
  for (auto &[s, n] : c)
    if (g_done[s] < n) return true;
  return false;
}
void merge(Clock &a, const Clock &b) {
  for (auto &[s, n] : b) a[s] = std::max(a[s], n);
}
void work(Stream *s) { ++s->clock[s->id]; }
bool any_capture() {
  for (Stream *s : g_streams)
    if (s->capturing) return true;
  return false;
}

void segments(const unsigned char *base, const SegJob *jobs, int32_t nj, double cut, int32_t *len) {
  for (int k = 0; k < nj; ++k) {
    const SegJob &j = jobs[k];
    const double *bx = (const double *)(base + j.bra_x), *kx = (const double *)(base + j.ket_x);
    const int32_t *bg = (const int32_t *)(base + j.bra_group), *gb = (const int32_t *)(base + j.group_begin),
                  *ge = (const int32_t *)(base + j.group_end);
    for (int i = 0; i < j.nbra; ++i)
      for (int g = 0; g < j.ngroup; ++g) {
        int a = gb[g], lim = ge[g];
        while (a < ge[g] && (j.cmp == CMP_NONE || (j.cmp == CMP_GT ? bx[i] * kx[a] > cut : !(bx[i] * kx[a] < cut)))) ++a;
        if (j.diag && g > bg[i]) a = gb[g];
        if (j.diag && g == bg[i]) lim = i + 1;
        len[j.len0 + (int64_t)i * j.ngroup + g] = std::max(0, std::min(a, lim) - gb[g]);
      }
  }
}

std::string tile_lengths(const ClassDev &c) {
  int32_t mx = 0;
  int64_t sum = 0;
  for (int i = 0; i < c.ntile; ++i) mx = std::max(mx, c.tiles[i].n), sum += c.tiles[i].n;
  return "tiles=" + std::to_string(c.ntile) + " longest=" + std::to_string(mx) + " quartets=" + std::to_string(sum) +
         " share=" + std::to_string(c.q_end - c.q_begin);
}

}  // namespace

extern "C" {

// ---- what the tests look at
const char *host_log() { return g_log.c_str(); }
void host_clear() { g_log.clear(); }
size_t host_bytes() { return g_bytes; }
size_t host_peak() { return g_peak; }
void host_clear_peak() { g_peak = g_bytes; }
// allocations of at least n bytes fail (0: none)
void host_fail(size_t n) { g_fail = n; }
int host_id(Stream *s) { return s->id; }
// whether the work issued so far on a comes before what b issues next
int host_before(Stream *a, Stream *b) { return b->clock[a->id] >= a->clock[a->id]; }
int host_in_flight(Stream *s) { return in_flight(s->clock); }
// work items of s that nothing has waited for
long host_outstanding(Stream *s) { return s->clock[s->id] - g_done[s->id]; }

// ---- the runtime
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (any_capture() && g_mode != hipStreamCaptureModeRelaxed) return err(hipErrorStreamCaptureUnsupported);
  if (g_fail && n >= g_fail) return log("malloc failed %zu", n), err(hipErrorOutOfMemory);
  *p = malloc(n);
  g_mem[*p] = n;
  g_bytes += n;
  g_peak = std::max(g_peak, g_bytes);
  log("malloc %zu", n);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  for (Stream *s : g_streams) done(s->clock);  // waits for the device
  g_bytes -= g_mem.at(p);
  g_mem.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  memcpy(d, s, n);
  work((Stream *)st);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  auto *n = new Stream{g_next++};
  g_streams.insert(n);
  *s = (hipStream_t)n;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  done(((Stream *)s)->clock);
  g_streams.erase((Stream *)s);
  delete (Stream *)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  auto *s = (Stream *)st;
  if (s->capturing) return err(hipErrorStreamCaptureUnsupported);
  done(s->clock);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t ev, unsigned) {
  auto *s = (Stream *)st;
  auto *e = (Event *)ev;
  if (e->captured && !s->capturing) return err(hipErrorCapturedEvent);
  if (!s->capturing) merge(s->clock, e->clock);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t) new Event, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (Event *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t st) {
  auto *e = (Event *)ev;
  auto *s = (Stream *)st;
  e->recorded = true;
  e->captured = s->capturing;
  if (!s->capturing) e->clock = s->clock;
  e->last = s->last;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t ev) {
  auto *e = (Event *)ev;
  if (e->captured) return err(hipErrorCapturedEvent);
  done(e->clock);
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t ev) {
  auto *e = (Event *)ev;
  if (e->captured) return err(hipErrorCapturedEvent);
  return in_flight(e->clock) ? hipErrorNotReady : hipSuccess;
}
// row forms take half the time of the others, lane row forms of 512 threads a
// tenth less
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t b) {
  const std::string &k = ((Event *)b)->last;
  if (((Event *)b)->captured) return err(hipErrorCapturedEvent);
  *ms = k.find("eri_row") != k.npos || k.find("eri_split") != k.npos ? 0.01f : 0.02f;
  if (k.find("eri_row") != k.npos && k.find(" 512") != k.npos) *ms *= 0.9f;
  return hipSuccess;
}
static thread_local struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t st;
} g_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st) {
  g_call = {g, b, lds, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st) {
  *g = g_call.grid, *b = g_call.block, *lds = g_call.lds, *st = g_call.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t st) {
  Dl_info info{};
  dladdr(f, &info);
  const std::string name = info.dli_sname ? info.dli_sname : "?";
  auto *s = (Stream *)st;
  std::string more;
  if (name.find("segment_lengths") != name.npos)
    segments(*(const unsigned char **)args[0], *(const SegJob **)args[1], *(int32_t *)args[2], *(double *)args[3],
             *(int32_t **)args[4]);
  if (name.find("eri_row_kernel") != name.npos || name.find("eri_split_kernel") != name.npos) {
    const ClassDev &c = *(const ClassDev *)args[0];
    more = " " + tile_lengths(c) + (c.ntile == (int)grid.x ? "" : " GRID");
  }
  if (name.find("eri_shared_") != name.npos) {
    const SharedArgs &sa = *(const SharedArgs *)args[0];
    const ClassDev *cds = *(const ClassDev **)args[1];
    const char launch = name[name.find("eri_shared_") + 11];
    more = std::string(" launch=") + launch;
    for (int k = 0; k < sa.n; ++k) {
      more += " [class=" + std::to_string(sa.cls[k]) + " transposed=" + std::to_string(cds[sa.cls[k]].transposed);
      if (launch < '0' + kSharedRowLaunches) more += " " + tile_lengths(cds[sa.cls[k]]);
      more += "]";
    }
  }
  if (name.find("build_begin") != name.npos) {
    // records of the primitive pairs that a kernel reads of a pair: at least the
    // first must be there
    const BuildArgs &ba = *(const BuildArgs *)args[1];
    const int64_t np = (int64_t)(g_mem.at((void *)ba.pairs) / sizeof(PairRec)),
                  nr = (int64_t)(g_mem.at((void *)ba.prims) / sizeof(PrimRec));
    int64_t empty = 0, past = 0;
    for (int64_t p = 0; p < np; ++p) {
      const PairRec &r = ba.pairs[p];
      empty += r.nprim == 0;
      past += r.prim_off < 0 || r.prim_off + (int64_t)std::max(r.nprim - 1, 0) * r.prim_stride >= nr;
    }
    char b[160];
    snprintf(b, sizeof b, " pairs=%ld records=%ld empty=%ld past=%ld Jp=%p", (long)np, (long)nr, (long)empty, (long)past,
             (void *)ba.Jp);
    more = b;
  }
  log("launch %s stream=%d captured=%d grid=%u block=%u%s", name.c_str(), s->id, s->capturing, grid.x, block.x,
      more.c_str());
  if (s->capturing)
    s->deps = {++g_node};
  else
    work(s);
  s->last = name + " " + std::to_string(block.x);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
  *c = ((Stream *)s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
  std::swap(*m, g_mode);
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  ((Stream *)s)->capturing = true;
  ((Stream *)s)->deps.clear();
  log("capture stream=%d", ((Stream *)s)->id);
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  ((Stream *)s)->capturing = false;
  *g = (hipGraph_t)malloc(8);
  return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t st, hipStreamCaptureStatus *c, unsigned long long *, hipGraph_t *,
                                      const hipGraphNode_t **d, size_t *n) {
  auto *s = (Stream *)st;
  *c = s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  *n = 0;
  for (size_t k : s->deps) g_deps[(*n)++] = (hipGraphNode_t)k;
  *d = g_deps;
  return hipSuccess;
}
hipError_t hipStreamUpdateCaptureDependencies(hipStream_t st, hipGraphNode_t *d, size_t n, unsigned) {
  auto *s = (Stream *)st;
  if (!s->capturing) return err(hipErrorIllegalState);
  s->deps.clear();
  for (size_t i = 0; i < n; ++i) s->deps.insert((size_t)d[i]);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = (hipGraphExec_t) new Exec{g_next++};
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t ge, hipStream_t st) {
  auto *e = (Exec *)ge;
  auto *s = (Stream *)st;
  if (!s->capturing) {
    work(s);
    e->after = s->clock;
  }
  s->last = "graph";
  log("replay graph=%d stream=%d captured=%d", e->id, s->id, s->capturing);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return free(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t ge) {
  auto *e = (Exec *)ge;
  log("destroy graph=%d in_flight=%d", e->id, in_flight(e->after));
  delete e;
  return hipSuccess;
}
}
