// A HIP runtime for the host code alone, without a device: the library's host
// objects are linked against it and driven through the C ABI.  Device memory is
// host memory, copies are made at once and checked against their allocations, a
// kernel launch is counted and does nothing, except that the few results the
// host code branches on (list check, control slots of a recorded solve) are
// written as the driver sets them.  Streams, events and graphs are modelled far
// enough to check their use: what is captured is joined, nothing that a capture
// forbids is called inside one, a graph is destroyed once and not while a
// launch of it is outstanding.  What breaks a rule is kept as text for the
// driver (stub_faults).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "nb_kern.h"

namespace {

std::string faults;
void fault(const std::string &what) { faults += what + "\n"; }

struct Capture;
struct Stream {
  bool live = true;
  Capture *cap = nullptr;
  std::map<Stream *, long> seen;            // capture: operations of each stream that this one waits for
  std::set<struct Exec *> outstanding;      // graphs launched since the last synchronisation
};
struct Event {
  bool live = true;
  Capture *cap = nullptr;
  bool stale = false;                       // recorded in a capture that has ended
  std::map<Stream *, long> seen;
  std::set<struct Exec *> outstanding;
  Stream *on = nullptr;
};
struct Op {
  const void *func = nullptr;               // a kernel, or a copy
  std::vector<void *> pin;                  // k_pack_outputs: its destination
  void *dst = nullptr;
  const void *src = nullptr;
  size_t bytes = 0;
};
struct Graph { std::vector<Op> ops; };
struct Capture {
  Stream *origin;
  Graph *graph;
  std::map<Stream *, long> count;
};
struct Exec {
  Graph graph;
  long launches = 0;
};

std::map<char *, size_t> device, pinned;
std::vector<long> sizes;                    // of the allocations since the last reset
// (registered by the constructors of the other objects, before this one's)
std::map<const void *, std::string> &kernels() {
  static auto *m = new std::map<const void *, std::string>();
  return *m;
}
std::set<Stream *> streams;
std::set<Event *> events;
std::set<Graph *> graphs;
std::set<Exec *> execs;
Capture *active = nullptr;

// set by the driver
long fail_bytes = 0;                        // allocations of this many bytes or more fail (0: none do)
long free_bytes = 1l << 38;                 // free device memory, as hipMemGetInfo tells it
int moved = 0, reject = 0, iterations = 1;

// counted for the driver
enum { C_LAUNCHES, C_CAPTURES, C_INSTANTIATED, C_REPLAYS, C_DESTROYED, C_UNUSED, C_FAILED, C_LDS, C_LIVE, C_N };
long counts[C_N];

struct Config { dim3 grid, block; size_t lds; hipStream_t stream; } config;

bool inside(const std::map<char *, size_t> &m, const void *p, size_t bytes) {
  auto it = m.upper_bound((char *)p);
  if (it == m.begin()) return false;
  --it;
  return (char *)p + bytes <= it->first + it->second;
}

void forbidden(const char *call) {
  if (active) fault(std::string(call) + " inside a capture");
}

Stream *of(hipStream_t s) {
  Stream *p = (Stream *)s;
  if (!p || !streams.count(p)) {
    fault("a stream that does not exist");
    return *streams.begin();
  }
  return p;
}

void add(Stream *s, const Op &op) {
  if (s->cap) {
    s->cap->graph->ops.push_back(op);
    s->seen[s] = ++s->cap->count[s];
  } else if (active) {
    fault("work on a stream outside the capture");
  }
}

void copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
  const bool to = kind == hipMemcpyHostToDevice || kind == hipMemcpyDeviceToDevice;
  const bool from = kind == hipMemcpyDeviceToHost || kind == hipMemcpyDeviceToDevice;
  if (to && !inside(device, dst, bytes)) return fault("copy past the end of a device allocation (write)");
  if (from && !inside(device, src, bytes)) return fault("copy past the end of a device allocation (read)");
  memmove(dst, src, bytes);
}

// the results that the host code reads back
void run(const Op &op) {
  if (!op.func) {
    memmove(op.dst, op.src, op.bytes);
  } else if (op.pin.size()) {
    double *pin = (double *)op.pin[0];
    memset(pin, 0, sizeof(double) * P_NSLOT);
    ((int32_t *)(pin + P_FLAGS))[3] = reject;
    pin[P_SCAL + S_DONE] = 1.0;
    pin[P_SCAL + S_ITER] = iterations;
  }
}

hipError_t launch(const void *func, void **args, size_t lds, hipStream_t stream) {
  counts[C_LAUNCHES]++;
  if ((long)lds > counts[C_LDS]) counts[C_LDS] = (long)lds;
  auto it = kernels().find(func);
  if (it == kernels().end()) {
    fault("an unknown kernel");
    return hipErrorInvalidValue;
  }
  Op op;
  op.func = func;
  if (it->second.find("k_pack_outputs") != std::string::npos) op.pin.push_back(*(void **)args[6]);
  if (it->second.find("k_max_disp") != std::string::npos && !active) (*(int32_t **)args[4])[3] = moved;
  Stream *s = of(stream);
  add(s, op);
  if (!s->cap) run(op);
  return hipSuccess;
}

hipError_t allocate(std::map<char *, size_t> &m, void **p, size_t bytes) {
  forbidden("an allocation");
  if (fail_bytes && (long)bytes >= fail_bytes) {
    counts[C_FAILED]++;
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  *p = calloc(1, bytes ? bytes : 1);
  m[(char *)*p] = bytes;
  sizes.push_back((long)bytes);
  counts[C_LIVE]++;
  return hipSuccess;
}

hipError_t release(std::map<char *, size_t> &m, void *p) {
  forbidden("a free");
  if (!p) return hipSuccess;
  if (!m.erase((char *)p)) {
    fault("a free of memory that is not allocated");
    return hipErrorInvalidValue;
  }
  for (Stream *s : streams) s->outstanding.clear();   // the runtime waits for the device
  free(p);
  counts[C_LIVE]--;
  return hipSuccess;
}

template <typename T> hipError_t make(std::set<T *> &set, void *out) {
  T *p = new T();
  set.insert(p);
  counts[C_LIVE]++;
  *(T **)out = p;
  return hipSuccess;
}

template <typename T> bool drop(std::set<T *> &set, void *p, const char *what) {
  if (!set.erase((T *)p)) {
    fault(std::string(what) + " destroyed that does not exist");
    return false;
  }
  counts[C_LIVE]--;
  return true;
}

}  // namespace

extern "C" {

void stub_set(long fail_at, int mv, int rj, int it) {
  fail_bytes = fail_at;
  moved = mv;
  reject = rj;
  iterations = it;
}
void stub_fault(const char *what) { fault(what); }
void stub_free(long bytes) { free_bytes = bytes; }
void stub_counts(long *out) { memcpy(out, counts, sizeof(counts)); }
void stub_reset_counts() {
  const long live = counts[C_LIVE];
  memset(counts, 0, sizeof(counts));
  counts[C_LIVE] = live;
  sizes.clear();
}
long stub_allocations(long *out, long most) {
  for (long i = 0; i < most && i < (long)sizes.size(); i++) out[i] = sizes[i];
  return (long)sizes.size();
}
const char *stub_faults() { return faults.c_str(); }
void stub_forget() { faults.clear(); }

void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  kernels()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  config = Config{grid, block, lds, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  *grid = config.grid;
  *block = config.block;
  *lds = config.lds;
  *stream = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t stream) {
  if (!grid.x || !grid.y || !grid.z || block.x * block.y * block.z > 1024) fault("a launch of impossible shape: " + kernels()[f]);
  return launch(f, args, lds, stream);
}
hipError_t hipExtLaunchKernel(const void *f, dim3, dim3, void **args, size_t lds, hipStream_t stream, hipEvent_t,
                              hipEvent_t, int) {
  return launch(f, args, lds, stream);
}

const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 163840;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char *scratch = nullptr;
  if (!scratch) {
    scratch = (char *)calloc(1, (size_t)NB_BATCH_SCRATCH_MIB << 20);
    device[scratch] = (size_t)NB_BATCH_SCRATCH_MIB << 20;
  }
  *p = scratch;
  return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) { return allocate(device, p, bytes); }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  forbidden("hipMemGetInfo");
  *f = (size_t)free_bytes;
  *t = (size_t)1 << 38;
  return hipSuccess;
}
hipError_t hipFree(void *p) { return release(device, p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(pinned, p, bytes); }
hipError_t hipHostFree(void *p) { return release(pinned, p); }
hipError_t hipMemset(void *p, int v, size_t bytes) {
  forbidden("hipMemset");
  if (!inside(device, p, bytes)) fault("hipMemset past the end of an allocation");
  else memset(p, v, bytes);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t bytes, hipStream_t s) {
  if (of(s)->cap) fault("hipMemsetAsync in a captured graph");
  return hipMemset(p, v, bytes);
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
  forbidden("hipMemcpy");
  copy(dst, src, bytes, kind);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t stream) {
  Stream *s = of(stream);
  Op op;
  op.dst = dst;
  op.src = src;
  op.bytes = bytes;
  add(s, op);
  if (!s->cap) {
    copy(dst, src, bytes, kind);
  } else {
    if (kind == hipMemcpyDeviceToHost && !inside(pinned, dst, bytes)) fault("a captured copy to memory that is not pinned");
    if (kind == hipMemcpyHostToDevice && !inside(pinned, src, bytes)) fault("a captured copy from memory that is not pinned");
  }
  return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t *s) { return make(streams, s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(streams, s); }
hipError_t hipStreamDestroy(hipStream_t s) {
  if (of(s)->cap) fault("a capturing stream destroyed");
  drop(streams, s, "a stream");
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t stream) {
  forbidden("hipStreamSynchronize");
  of(stream)->outstanding.clear();
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return make(events, e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(events, e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  drop(events, e, "an event");
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t stream) {
  Event *e = (Event *)ev;
  Stream *s = of(stream);
  if (active && !s->cap) fault("an event recorded outside the capture");
  e->cap = s->cap;
  e->stale = false;
  e->seen = s->seen;
  e->outstanding = s->outstanding;
  e->on = s;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t stream, hipEvent_t ev, unsigned) {
  Event *e = (Event *)ev;
  Stream *s = of(stream);
  if (e->stale) fault("a wait for an event of a capture that has ended");
  if (e->cap) {
    if (s->cap && s->cap != e->cap) fault("a wait across captures");
    s->cap = e->cap;
    e->cap->count[s];
    for (auto &q : e->seen) {
      long &v = s->seen[q.first];
      if (q.second > v) v = q.second;
    }
  } else if (s->cap) {
    fault("a capturing stream waits for an event outside the capture");
  } else {
    s->outstanding.insert(e->outstanding.begin(), e->outstanding.end());
  }
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t ev) {
  forbidden("hipEventSynchronize");
  Event *e = (Event *)ev;
  if (e->on && streams.count(e->on))
    for (Exec *x : e->outstanding) e->on->outstanding.erase(x);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t stream, hipStreamCaptureMode) {
  forbidden("hipStreamBeginCapture");
  Stream *s = of(stream);
  active = new Capture{s, new Graph(), {}};
  s->cap = active;
  s->seen.clear();
  counts[C_CAPTURES]++;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t stream, hipGraph_t *out) {
  Stream *s = of(stream);
  *out = nullptr;
  if (!active || active->origin != s) {
    fault("hipStreamEndCapture without its capture");
    return hipErrorInvalidValue;
  }
  for (auto &q : active->count)
    if (q.first != s && s->seen[q.first] < q.second) fault("a captured stream is not joined");
  for (Stream *t : streams)
    if (t->cap == active) {
      t->cap = nullptr;
      t->seen.clear();
    }
  for (Event *e : events)
    if (e->cap == active) {
      e->cap = nullptr;
      e->stale = true;
    }
  graphs.insert(active->graph);
  counts[C_LIVE]++;
  *(Graph **)out = active->graph;
  delete active;
  active = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *out, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  forbidden("hipGraphInstantiate");
  make(execs, out);
  (*(Exec **)out)->graph = *(Graph *)g;
  counts[C_INSTANTIATED]++;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  if (drop(graphs, g, "a graph")) delete (Graph *)g;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t stream) {
  forbidden("hipGraphLaunch");
  Exec *e = (Exec *)x;
  if (!execs.count(e)) {
    fault("a graph launched that does not exist");
    return hipErrorInvalidValue;
  }
  counts[C_REPLAYS]++;
  e->launches++;
  of(stream)->outstanding.insert(e);
  for (const Op &op : e->graph.ops) run(op);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  Exec *e = (Exec *)x;
  for (Stream *s : streams)
    if (s->outstanding.count(e)) fault("a graph destroyed while a launch of it is outstanding");
  if (drop(execs, e, "an executable graph")) {
    counts[C_DESTROYED]++;
    if (!e->launches) counts[C_UNUSED]++;
    delete e;
  }
  return hipSuccess;
}

}  // extern "C"
