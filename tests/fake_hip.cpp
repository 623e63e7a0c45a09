// fake_hip.cpp -- the HIP runtime calls of libdlbc_hip.so on host memory, for
// tests of its host code on a machine without a GPU.
//
// Loaded with RTLD_GLOBAL before the library, its functions take the place of
// the runtime's.  Memory is the host's and copies are made at once; a kernel
// launch is counted under the kernel's (mangled) name and does nothing but what
// the one-launch step does to its flags.  Calls are counted, can be made to fail,
// and remember the device that was current.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace {

std::mutex mu;
std::map<std::string, int64_t> calls, launches;
struct Failure {
  int64_t in;  // calls until it; 0: every call
  int code;
};
std::map<std::string, Failure> failures;
std::map<const void *, std::string> kernels;
std::map<const void *, int> device_of;  // of allocations, events and streams
std::map<int64_t, int64_t> live;        // allocations and events by device
thread_local int current = 0;
thread_local int last_error = 0;

// Counts a call; its result: 0, or the code it was told to fail with.
int called(const char *name) {
  std::lock_guard<std::mutex> lock(mu);
  ++calls[name];
  auto f = failures.find(name);
  if (f == failures.end()) return 0;
  const Failure now = f->second;
  if (now.in > 1) {
    --f->second.in;
    return 0;
  }
  if (now.in == 1) failures.erase(f);
  return last_error = now.code;
}

void *made(void *p) {
  std::lock_guard<std::mutex> lock(mu);
  device_of[p] = current;
  ++live[current];
  return p;
}

int gone(void *p) {
  if (!p) return 0;
  {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = device_of.find(p);
    if (it == device_of.end()) return 1;
    --live[it->second];
    device_of.erase(it);
  }
  std::free(p);
  return 0;
}

// The flags of the one-launch step (SplitPlan, the seventh argument of its
// kernels): all of a launch's own set are down when it starts and up when it has
// ended, and those of the other set are down then.
struct Plan {
  const int32_t *order;
  uint8_t *flags;
  int nflag, set, polls;
};
int64_t flags_up = 0;  // launches that started with some of their flags up
void run_plan(const Plan &q) {
  uint8_t *own = q.flags + (int64_t)q.set * q.nflag, *other = q.flags + (int64_t)(q.set ^ 1) * q.nflag;
  for (int k = 0; k < q.nflag; ++k)
    if (own[k]) {
      ++flags_up;
      break;
    }
  std::memset(own, 1, q.nflag);
  std::memset(other, 0, q.nflag);
}
bool one_launch(const std::string &name) {  // the last template argument: true
  return name.find("split_collide") != std::string::npos &&
         name.find("Lb1EEEv") != std::string::npos;
}
struct Graph {
  std::vector<Plan> plans;
  int64_t nodes = 0;
};
std::map<void *, Graph> capturing;  // by stream
int64_t graph_nodes = 0;            // kernels of the graph launched last

// Pinned memory that copies queued on a stream still use: until the stream, or an
// event recorded after them by their thread, was waited for.
std::set<const void *> pinned;
std::map<const void *, void *> busy;  // pinned memory -> stream
std::map<const void *, const void *> recorded_after;  // event -> pinned memory
thread_local const void *last_used = nullptr;
int64_t busy_used = 0;
void uses(const void *p, void *stream) {
  if (!pinned.count(p)) return;
  if (busy.count(p)) ++busy_used;
  busy[p] = stream;
  last_used = p;
}
void waited(void *stream) {
  for (auto it = busy.begin(); it != busy.end();)
    it = it->second == stream ? busy.erase(it) : std::next(it);
}

struct Dim3 {
  uint32_t x, y, z;
};
struct Call {
  Dim3 grid, block;
  size_t shared;
  void *stream;
};
thread_local std::vector<Call> pushed;

}  // namespace

extern "C" {

// ---- what a test asks ------------------------------------------------------------
int64_t fake_hip_calls(const char *name) {
  std::lock_guard<std::mutex> lock(mu);
  return calls[name];
}
// Launches of the kernels whose mangled name holds `part`.
int64_t fake_hip_launches(const char *part) {
  std::lock_guard<std::mutex> lock(mu);
  int64_t n = 0;
  for (const auto &k : launches)
    if (k.first.find(part) != std::string::npos) n += k.second;
  return n;
}
// Allocations and events that are alive on a device.
int64_t fake_hip_live(int device) {
  std::lock_guard<std::mutex> lock(mu);
  return live[device];
}
// Launches of the one-launch step that started with some of their flags up.
int64_t fake_hip_flags_up() {
  std::lock_guard<std::mutex> lock(mu);
  return flags_up;
}
int64_t fake_hip_graph_nodes() {
  std::lock_guard<std::mutex> lock(mu);
  return graph_nodes;
}
// Pinned memory used again or freed while a copy may be under way in it.
int64_t fake_hip_busy_used() {
  std::lock_guard<std::mutex> lock(mu);
  return busy_used;
}
// The nth call of `name` from now on returns `code`, or every call (nth 0).
void fake_hip_fail(const char *name, int nth, int code) {
  std::lock_guard<std::mutex> lock(mu);
  failures[name] = {nth, code};
}

// ---- the runtime -------------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, Dim3 *, Dim3 *, int *) {
  std::lock_guard<std::mutex> lock(mu);
  kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
  pushed.push_back({grid, block, shared, stream});
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
  const Call c = pushed.back();
  pushed.pop_back();
  *grid = c.grid;
  *block = c.block;
  *shared = c.shared;
  *stream = c.stream;
  return 0;
}
int hipLaunchKernel(const void *host, Dim3, Dim3, void **args, size_t, void *stream) {
  if (const int e = called("hipLaunchKernel")) return e;
  std::lock_guard<std::mutex> lock(mu);
  const std::string &name = kernels[host];
  ++launches[name];
  const auto c = capturing.find(stream);
  if (c != capturing.end()) ++c->second.nodes;
  if (one_launch(name)) {
    const Plan q = *static_cast<const Plan *>(args[6]);
    if (c != capturing.end())
      c->second.plans.push_back(q);
    else
      run_plan(q);
  }
  return 0;
}
int hipLaunchCooperativeKernel(const void *host, Dim3 grid, Dim3 block, void **args,
                               unsigned shared, void *stream) {
  return hipLaunchKernel(host, grid, block, args, shared, stream);
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 1;
  return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
  *v = 256;
  return 0;
}
int hipGetLastError() {
  if (const int e = called("hipGetLastError")) {
    last_error = 0;
    return e;
  }
  const int e = last_error;
  last_error = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e ? "planned failure" : "no error"; }
int hipSetDevice(int d) {
  if (const int e = called("hipSetDevice")) return e;
  current = d;
  return 0;
}
int hipGetDevice(int *d) {
  *d = current;
  return 0;
}
int hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (const int e = called("hipMalloc")) return e;
  *p = made(std::calloc(n ? n : 1, 1));
  return 0;
}
int hipFree(void *p) { return gone(p); }
int hipHostMalloc(void **p, size_t n, unsigned) {
  *p = nullptr;
  if (const int e = called("hipHostMalloc")) return e;
  *p = made(std::calloc(n, 1));
  std::lock_guard<std::mutex> lock(mu);
  pinned.insert(*p);
  return 0;
}
int hipHostFree(void *p) {
  if (const int e = called("hipHostFree")) return e;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (busy.count(p)) ++busy_used;
    pinned.erase(p);
  }
  return gone(p);
}
int hipGetSymbolAddress(void **p, const void *) {
  static double room[1 << 20];
  *p = room;
  return 0;
}
int hipMemcpy(void *to, const void *from, size_t n, int) {
  if (const int e = called("hipMemcpy")) return e;
  std::memcpy(to, from, n);
  return 0;
}
int hipMemcpyAsync(void *to, const void *from, size_t n, int, void *stream) {
  if (const int e = called("hipMemcpyAsync")) return e;
  std::memcpy(to, from, n);
  std::lock_guard<std::mutex> lock(mu);
  uses(to, stream);
  uses(from, stream);
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t n, void *) {
  if (const int e = called("hipMemsetAsync")) return e;
  std::memset(p, v, n);
  return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned) {
  *s = std::calloc(1, 8);
  return 0;
}
int hipStreamDestroy(void *s) {
  std::free(s);
  return 0;
}
int hipStreamSynchronize(void *stream) {
  if (const int e = called("hipStreamSynchronize")) return e;
  std::lock_guard<std::mutex> lock(mu);
  waited(stream);
  return 0;
}
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreateWithFlags(void **e, unsigned) {
  *e = nullptr;
  if (const int err = called("hipEventCreateWithFlags")) return err;
  *e = made(std::calloc(1, 8));
  return 0;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { return gone(e); }
int hipEventRecord(void *event, void *) {
  if (const int e = called("hipEventRecord")) return e;
  std::lock_guard<std::mutex> lock(mu);
  recorded_after[event] = last_used;
  return 0;
}
int hipEventSynchronize(void *event) {
  if (const int e = called("hipEventSynchronize")) return e;
  std::lock_guard<std::mutex> lock(mu);
  busy.erase(recorded_after[event]);
  return 0;
}
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 1.0f;
  return 0;
}
int hipStreamBeginCapture(void *stream, int) {
  if (const int e = called("hipStreamBeginCapture")) return e;
  std::lock_guard<std::mutex> lock(mu);
  capturing[stream] = Graph{};
  return 0;
}
int hipStreamEndCapture(void *stream, void **g) {
  *g = nullptr;
  const int e = called("hipStreamEndCapture");
  std::lock_guard<std::mutex> lock(mu);
  if (!e) *g = new Graph(capturing[stream]);
  capturing.erase(stream);
  return e;
}
int hipGraphInstantiate(void **x, void *g, void *, char *, size_t) {
  *x = nullptr;
  if (const int e = called("hipGraphInstantiate")) return e;
  *x = new Graph(*static_cast<Graph *>(g));
  return 0;
}
int hipGraphDestroy(void *g) {
  delete static_cast<Graph *>(g);
  return 0;
}
int hipGraphExecDestroy(void *x) {
  delete static_cast<Graph *>(x);
  return 0;
}
int hipGraphLaunch(void *x, void *) {
  if (const int e = called("hipGraphLaunch")) return e;
  std::lock_guard<std::mutex> lock(mu);
  graph_nodes = static_cast<Graph *>(x)->nodes;
  for (const Plan &q : static_cast<Graph *>(x)->plans) run_plan(q);
  return 0;
}

}  // extern "C"
