// The library's host code against a stand-in for the HIP runtime (CPU only).
//
// This program defines the runtime functions that libqwen_megakernel.so calls and then loads the
// library, which binds to them. Nothing runs on a GPU: every operation is noted with the operations
// it must follow (its stream's last one, an event's, the cooperative queue's), a captured stream
// notes graph nodes, and a replay adds them as hipGraphLaunch would. After each scenario it checks
// what the kernels rely on:
//  * every kernel of the library follows all earlier ones, whatever their streams, replayed or not
//    (the workspaces are shared, and two grids whose workgroups wait for each other must not share
//    the chip);
//  * every grid was checked to be resident at once, and a grid that needs the whole chip does not go
//    to a queue that is restricted to some of its CUs.
// usage: launch_order_check <library> <scenario>; exits 0 if the scenario holds.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <mutex>
#include <vector>

#include "qwen_megakernel.h"

namespace {

struct Op {
  std::string what;
  std::vector<int> preds;
  bool ours;  // a kernel of the library that uses the workspaces
};
struct Node {
  enum Kind { KERNEL, COOP, WAIT, RECORD } kind;
  std::string what;
  bool ours;
  hipEvent_t event;
};
struct Stream {
  int tail = -1;
  bool capturing = false, capture_unknown = false;
  uint32_t mask = 0xffffffffu;  // every word of its CU mask
  std::vector<Node> graph;
  Node pending;  // an explicitly added node, until the capture's dependencies are set to it
};
std::recursive_mutex mu;
std::vector<Op> ops;
std::map<hipStream_t, Stream> streams;
std::map<hipEvent_t, int> events;
std::map<const void*, std::string> names;
std::map<const void*, int> checked;  // kernel -> workgroups per CU it was found to fit
std::string unfit;                   // a kernel whose name holds this fits no CU
int coop_tail = -1, done = 0, grids = 0, bad = 0;
dim3 cfg_grid, cfg_block;
hipStream_t cfg_stream;

#define LOCK std::lock_guard<std::recursive_mutex> lock(mu)
void complain(const std::string& s) {
  ++bad;
  fprintf(stderr, "launch order: %s\n", s.c_str());
}
bool follows(int a, int b) {  // does op a follow op b?
  std::set<int> seen;
  std::vector<int> todo{a};
  while (!todo.empty()) {
    const int i = todo.back();
    todo.pop_back();
    if (i == b) return true;
    if (i < b || !seen.insert(i).second) continue;
    for (int p : ops[i].preds) todo.push_back(p);
  }
  return false;
}
int add(hipStream_t s, const std::string& what, bool ours, bool coop, int also = -1) {
  Op o{what, {}, ours};
  for (int p : {streams[s].tail, coop ? coop_tail : -1, also})
    if (p >= 0) o.preds.push_back(p);
  ops.push_back(o);
  const int id = (int)ops.size() - 1;
  streams[s].tail = id;
  if (coop) coop_tail = id;
  if (ours)
    for (int k = done; k < id; ++k)
      if (ops[k].ours && !follows(id, k)) complain(what + " may run beside " + ops[k].what + " (operation " + std::to_string(k) + ")");
  return id;
}
// a replay of what the stream captured
void replay(hipStream_t s) {
  LOCK;
  for (const Node& n : streams[s].graph) switch (n.kind) {
      case Node::KERNEL: add(s, n.what, n.ours, false); break;
      case Node::COOP: add(s, n.what, n.ours, true); break;
      case Node::WAIT: add(s, "wait", false, false, events.count(n.event) ? events[n.event] : -1); break;
      case Node::RECORD: events[n.event] = add(s, "record", false, false); break;
    }
}
std::string name_of(const void* k) { return names.count(k) ? names[k] : "?"; }
bool is_probe(const std::string& n) { return n.find("placement_probe") != std::string::npos; }
void resident(const void* k, int grid) {
  const std::string n = name_of(k);
  if (is_probe(n)) return;  // (its workgroups do not wait)
  ++grids;
  if (!checked.count(k)) complain(n + " was not checked to fit");
  else if (grid > checked[k] * 256) complain(n + " does not fit");
}

}  // namespace

// ---- the runtime ---------------------------------------------------------------------------
extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* m;
  return &m;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t s) {
  mu.lock();
  cfg_grid = g, cfg_block = b, cfg_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = cfg_grid, *b = cfg_block, *m = 0, *s = cfg_stream;
  mu.unlock();
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  p->cooperativeLaunch = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 100000, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char* m = (char*)aligned_alloc(256, 16 << 20);
  return *p = m, hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return *p = aligned_alloc(256, (n + 255) / 256 * 256), hipSuccess; }
hipError_t hipFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipDeviceSynchronize() {
  LOCK;
  done = (int)ops.size();
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipDeviceSynchronize(); }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* k, int threads, size_t) {
  LOCK;
  *n = !unfit.empty() && name_of(k).find(unfit) != std::string::npos ? 0 : threads <= 256 ? 2 : 1;
  checked[k] = *n;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  LOCK;
  if (streams[s].capture_unknown) return hipErrorStreamCaptureImplicit;
  *st = streams[s].capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipExtStreamGetCUMask(hipStream_t s, uint32_t n, uint32_t* m) {
  LOCK;
  for (uint32_t i = 0; i < n; ++i) m[i] = streams[s].mask;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  static char pool[64];
  static int used;
  return *e = (hipEvent_t)(pool + used++), hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  LOCK;
  if (streams[s].capturing) return hipErrorStreamCaptureIsolation;  // (orders nothing outside the graph)
  events[e] = add(s, "record", false, false);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  LOCK;
  if (streams[s].capturing) return hipErrorStreamCaptureIsolation;
  add(s, "wait", false, false, events.count(e) ? events[e] : -1);
  return hipSuccess;
}
// (a captured stream stands for its graph; its nodes are one chain)
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t s, hipStreamCaptureStatus* st, unsigned long long* id, hipGraph_t* g,
                                      const hipGraphNode_t** deps, size_t* n) {
  LOCK;
  *st = streams[s].capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  *id = 1, *g = (hipGraph_t)s, *deps = nullptr, *n = streams[s].graph.size();
  return hipSuccess;
}
hipError_t hipGraphAddEventWaitNode(hipGraphNode_t* node, hipGraph_t g, const hipGraphNode_t*, size_t n, hipEvent_t e) {
  LOCK;
  if (n != streams[(hipStream_t)g].graph.size()) return hipErrorInvalidValue;
  if (!events.count(e)) complain("a node waits for an event that was never recorded");
  streams[(hipStream_t)g].pending = {Node::WAIT, "wait", false, e};
  return *node = (hipGraphNode_t)g, hipSuccess;
}
hipError_t hipGraphAddEventRecordNode(hipGraphNode_t* node, hipGraph_t g, const hipGraphNode_t*, size_t n, hipEvent_t e) {
  LOCK;
  if (n != streams[(hipStream_t)g].graph.size()) return hipErrorInvalidValue;
  streams[(hipStream_t)g].pending = {Node::RECORD, "record", false, e};
  return *node = (hipGraphNode_t)g, hipSuccess;
}
hipError_t hipStreamUpdateCaptureDependencies(hipStream_t s, hipGraphNode_t* node, size_t n, unsigned flags) {
  LOCK;
  if (n != 1 || *node != (hipGraphNode_t)s || flags != hipStreamSetCaptureDependencies) return hipErrorInvalidValue;
  streams[s].graph.push_back(streams[s].pending);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* k, dim3, dim3, void**, size_t, hipStream_t s) {
  LOCK;
  if (streams[s].capture_unknown) return complain("a launch on a stream whose capture state is unknown"), hipSuccess;
  if (streams[s].capturing) streams[s].graph.push_back({Node::KERNEL, name_of(k), true, nullptr});
  else add(s, name_of(k), true, false);
  return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void* k, dim3 g, dim3, void** args, unsigned, hipStream_t s) {
  LOCK;
  const std::string n = name_of(k);
  if (streams[s].capture_unknown) return complain("a launch on a stream whose capture state is unknown"), hipSuccess;
  resident(k, (int)g.x);
  if (is_probe(n))
    for (unsigned w = 0; w < g.x; ++w) (*(unsigned**)args[0])[w] = (w + 6) % 8;
  if (streams[s].capturing) streams[s].graph.push_back({Node::COOP, n, !is_probe(n), nullptr});
  else add(s, n, !is_probe(n), true);
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void* k, dim3 g, dim3, void**, size_t, hipStream_t s, hipEvent_t start, hipEvent_t stop, int) {
  LOCK;
  if (streams[s].capture_unknown) return complain("a launch on a stream whose capture state is unknown"), hipSuccess;
  if (streams[s].capturing) return hipErrorStreamCaptureUnsupported;
  resident(k, (int)g.x);
  if (streams[s].mask != 0xffffffffu) complain(name_of(k) + " goes to a queue restricted to some CUs");
  const int id = add(s, name_of(k), true, false);
  if (start) events[start] = id;
  if (stop) events[stop] = id;
  return hipSuccess;
}
}  // extern "C"

// ---- calls and scenarios ------------------------------------------------------------------------
namespace {

void* buf() {
  static void* p = aligned_alloc(4096, 1 << 20);
  return p;
}
hipStream_t stream(int k) {
  static char s[8];
  return (hipStream_t)(k ? s + k : nullptr);
}
void* lib;
template <typename F>
F* fn(F*, const char* name) {
  F* f = (F*)dlsym(lib, name);
  if (!f) {
    fprintf(stderr, "no %s\n", name);
    exit(2);
  }
  return f;
}
#define CALL(f) fn(&f, #f)
const LDGLayerWeight* table() { return (const LDGLayerWeight*)buf(); }

int prefill(int n, int start, hipStream_t s) {
  void* b = buf();
  return CALL(qwen_prefill)((int*)b, n, b, table(), b, b, b, b, b, 2, start, 2048, 0.088f, s);
}
int generate(hipStream_t s) {
  void* b = buf();
  return CALL(qwen_generate_ex)(1, 4, nullptr, b, table(), b, b, b, b, b, b, b, (float*)b, (int*)b, nullptr, nullptr, 2, 0, 2048, 0.088f, s);
}
int sampled(float temperature, int top_k, float top_p, hipStream_t s) {
  void* b = buf();
  return CALL(qwen_generate_sampled)(1, 4, -1, b, table(), b, b, b, b, b, b, b, (float*)b, (int*)b, nullptr, 2, 0, 2048, 0.088f,
                                     temperature, top_k, top_p, 7, s);
}
int noalloc(hipStream_t s) {
  void* b = buf();
  return CALL(qwen_generate_nosync_noalloc)(1, 4, b, table(), b, b, b, b, b, b, b, b, b, b, b, b, b, b, (float*)b, b, b, (int*)b, 2, 0, 2048,
                                            0.088f, s);
}
int draw(hipStream_t s) { return CALL(qwen_sample)((float*)buf(), 5000, 0.8f, 0, 0.9f, 7, 3, (int*)buf(), s); }
int lm_head(hipStream_t s) { return CALL(qwen_lm_head_argmax)(buf(), buf(), (int*)buf(), nullptr, s); }
int mlp(hipStream_t s) { return CALL(qwen_mlp_block)(buf(), buf(), buf(), buf(), buf(), (float*)buf(), s); }

// every entry point and every build of the kernels once; the number of calls that failed
int all_calls(hipStream_t s, bool with_noalloc = true) {
  int f = 0;
  for (int n : {1, 17, 65, 129, 257, 513, 1025}) f += prefill(n, 0, s) != QWEN_OK;
  f += generate(s) != QWEN_OK;
  f += sampled(0.8f, 50, 0.9f, s) != QWEN_OK;   // top-k
  f += sampled(0.8f, 200, 0.9f, s) != QWEN_OK;  // the larger top-k, and top-p alone
  f += sampled(0.8f, 0, 1.0f, s) != QWEN_OK;    // temperature alone
  if (with_noalloc) f += noalloc(s) != QWEN_OK;
  f += (draw(s) != QWEN_OK) + (lm_head(s) != QWEN_OK) + (mlp(s) != QWEN_OK);
  return f;
}
void expect(bool ok, const char* what) {
  if (!ok) complain(std::string("expected: ") + what);
}

void eager() {
  for (int r = 0; r < 2; ++r)
    for (int k : {1, 2, 0}) expect(all_calls(stream(k)) == 0, "every call is accepted");
  expect(grids == 2 * 3 * 15, "every call launches its grid");
}
void threads() {
  expect(all_calls(stream(1)) == 0, "every call is accepted");
  std::thread a([] { for (int r = 0; r < 10; ++r) all_calls(stream(1)); }), b([] { for (int r = 0; r < 10; ++r) all_calls(stream(2)); });
  a.join();
  b.join();
}
// a captured call neither overtakes an eager one nor is overtaken, on the first replay and later ones
void captured() {
  expect(all_calls(stream(1)) == 0, "every call is accepted");
  streams[stream(2)].capturing = true;
  expect(prefill(61, 1400, stream(2)) == QWEN_OK && prefill(1500, 0, stream(2)) == QWEN_OK && lm_head(stream(2)) == QWEN_OK &&
             generate(stream(2)) == QWEN_OK && draw(stream(2)) == QWEN_OK,
         "a captured call is accepted");
  expect(mlp(stream(2)) == QWEN_ERR_LAUNCH && noalloc(stream(2)) == QWEN_ERR_ARG, "two entry points refuse capture");
  expect(all_calls(stream(1)) == 0, "eager calls beside a capture are accepted");
  streams[stream(2)].capturing = false;
  for (int r = 0; r < 3; ++r) {
    replay(stream(2));
    if (r) replay(stream(2));
    expect(prefill(61, 1400, stream(1)) == QWEN_OK, "a call after a replay");
    expect(generate(stream(3)) == QWEN_OK, "a call after a replay");
  }
}
// a queue restricted to some CUs cannot hold a grid that needs them all
void masked() {
  streams[stream(2)].mask = 0x0000ffffu;
  for (int r = 0; r < 2; ++r)
    for (int k : {2, 1, 2, 0}) expect(all_calls(stream(k)) == 0, "every call is accepted");
}
// a build that no longer fits is refused before anything is launched
void fits(const char* build) {
  unfit = build;
  expect(all_calls(stream(1)) == 15, "every call is refused");
  expect(grids == 0, "nothing is launched");
}
// where the runtime cannot say whether the stream is captured nothing is sent there
void unknown() {
  expect(all_calls(stream(1)) == 0, "every call is accepted");
  streams[stream(0)].capture_unknown = true;
  expect(all_calls(stream(0)) == 15, "every call is refused");
  streams[stream(0)].capture_unknown = false;
  expect(all_calls(stream(0)) == 0 && all_calls(stream(1)) == 0, "and later ones are accepted");
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  lib = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL);
  if (!lib) {
    fprintf(stderr, "%s\n", dlerror());
    return 2;
  }
  if (names.size() < 15) {
    fprintf(stderr, "the library did not bind to this program's runtime\n");
    return 2;
  }
  const std::string s = argv[2];
  if (s == "eager") eager();
  else if (s == "threads") threads();
  else if (s == "captured") captured();
  else if (s == "masked") masked();
  else if (s == "unknown") unknown();
  else if (s.rfind("fits:", 0) == 0) fits(s.c_str() + 5);
  else return 2;
  printf("%s: %d grids, %d operations, %d complaints\n", s.c_str(), grids, (int)ops.size(), bad);
  fflush(stdout);
  _Exit(bad ? 1 : 0);  // (the library's own exit handlers belong to the real runtime)
}
