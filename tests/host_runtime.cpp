// A stand-in for the HIP runtime on a machine without a GPU: "device" memory is
// host memory, kernels do not run, and what the library asks of the runtime is
// recorded (allocations, launches with their arguments, captured graphs).  Load
// it with RTLD_GLOBAL before the library, whose calls then bind to it.
#include <cxxabi.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

namespace {
constexpr int kOutOfMemory = 2, kUnsupported = 801;

struct Dim {
  uint32_t x, y, z;
};
struct Block {
  size_t bytes;
  int id;
  bool live;
};
struct Kernel {
  std::string name;
  std::vector<bool> pointer;  // per parameter
};
struct Node {  // a recorded launch, or (kernel null) a copy
  const Kernel* kernel;
  std::vector<void*> args;  // its pointer arguments (a copy's dst, src)
  std::vector<int> ids;     // the allocations they lay in (-1: in none)
  uint32_t grid;
  size_t bytes;
};

std::map<const void*, Kernel> kernels;
std::map<uintptr_t, Block> blocks;  // freed ones stay, so no address is used twice
std::vector<std::vector<Node>*> graphs;
std::vector<Node>* capture = nullptr;
std::map<std::string, int> launched;
std::map<std::string, std::vector<uint64_t>> lastArgs;
int failIn = 0, captures = 0, stale = 0;
size_t freeBytes = size_t(256) << 30;
Dim pushedGrid, pushedBlock;
size_t pushedShared;
void* pushedStream;

Block* find(const void* p) {
  auto it = blocks.upper_bound((uintptr_t)p);
  if (it == blocks.begin()) return nullptr;
  --it;
  return (uintptr_t)p < it->first + it->second.bytes ? &it->second : nullptr;
}

// kernel name without namespace and template arguments, and its parameters
Kernel describe(const char* mangled) {
  Kernel k;
  int st = 0;
  char* d = abi::__cxa_demangle(mangled, nullptr, nullptr, &st);
  std::string s = d ? d : mangled;
  free(d);
  size_t open = s.size(), depth = 0;
  while (open > 0) {  // the last parenthesised list
    open--;
    if (s[open] == ')') depth++;
    if (s[open] == '(' && --depth == 0) break;
  }
  std::string list = s.substr(open + 1, s.size() - open - 2), cur;
  int level = 0;
  for (char c : list + ",") {
    if (c == '<' || c == '(') level++;
    if (c == '>' || c == ')') level--;
    if (c == ',' && level == 0) {
      if (!cur.empty()) k.pointer.push_back(cur.back() == '*');
      cur.clear();
    } else {
      cur += c;
    }
  }
  std::string head = s.substr(0, open);
  size_t end = head.size();
  if (end && head[end - 1] == '>') {
    int lv = 0;
    do {
      end--;
      if (head[end] == '>') lv++;
      if (head[end] == '<') lv--;
    } while (lv && end);
  }
  head = head.substr(0, end);
  k.name = head.substr(head.rfind(':') + 1);
  k.name = k.name.substr(k.name.rfind(' ') + 1);
  return k;
}

// the one kernel with an effect: every sum a reduction ends with is 1, so that
// vectors have norms and solves go on
void effect(const Node& n) {
  if (n.kernel && n.kernel->name == "kFinalSum")
    for (uint32_t q = 0; q < n.grid; q++) static_cast<double*>(n.args[1])[q] = 1.0;
  if (!n.kernel) memcpy(n.args[0], n.args[1], n.bytes);
}

void submit(Node n) {
  for (void* p : n.args) {
    const Block* b = find(p);
    n.ids.push_back(b ? b->id : -1);
  }
  if (capture)
    capture->push_back(n);
  else
    effect(n);
}
}  // namespace

extern "C" {
// what tests ask
void fake_fail_in(int k) { failIn = k; }  // allocations fail from the k-th on (0: none)
void fake_set_free(uint64_t bytes) { freeBytes = bytes; }
int fake_stale() { return stale; }  // replayed arguments whose allocation was freed
int fake_captures() { return captures; }
int fake_launches(const char* name) { return launched[name]; }
uint64_t fake_last_arg(const char* name, int i) { return lastArgs[name].at(i); }
int fake_live() {
  int c = 0;
  for (auto& b : blocks) c += b.second.live;
  return c;
}

// the runtime
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, Dim*, Dim*,
                           int*) {
  kernels[host] = describe(device);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void* stream) {
  pushedGrid = grid;
  pushedBlock = block;
  pushedShared = shared;
  pushedStream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* shared, void** stream) {
  *grid = pushedGrid;
  *block = pushedBlock;
  *shared = pushedShared;
  *stream = pushedStream;
  return 0;
}
int hipLaunchKernel(const void* host, Dim grid, Dim, void** args, size_t, void*) {
  const Kernel& k = kernels.at(host);
  Node n{&k, {}, {}, grid.x, 0};
  std::vector<uint64_t> all;
  for (size_t i = 0; i < k.pointer.size(); i++) {
    uint64_t v = 0;
    memcpy(&v, args[i], k.pointer[i] ? 8 : 4);  // (of the others the first four bytes)
    all.push_back(v);
    if (k.pointer[i]) n.args.push_back((void*)v);
  }
  launched[k.name]++;
  lastArgs[k.name] = all;
  submit(n);
  return 0;
}
int hipMalloc(void** p, size_t bytes) {
  if (failIn == 1) return kOutOfMemory;
  if (failIn > 1) failIn--;
  static int ids = 0;
  *p = calloc(1, bytes ? bytes : 1);
  blocks[(uintptr_t)*p] = Block{bytes, ++ids, true};
  return 0;
}
int hipFree(void* p) {
  auto it = blocks.find((uintptr_t)p);
  if (it != blocks.end()) it->second.live = false;
  return 0;
}
int hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return 0;
}
int hipHostFree(void*) { return 0; }
int hipMemcpyAsync(void* dst, const void* src, size_t bytes, int, void*) {
  if (bytes) submit(Node{nullptr, {dst, const_cast<void*>(src)}, {}, 0, bytes});
  return 0;
}
int hipMemcpy(void* dst, const void* src, size_t bytes, int) {
  memcpy(dst, src, bytes);
  return 0;
}
int hipMemsetAsync(void* dst, int v, size_t bytes, void*) {
  if (bytes) memset(dst, v, bytes);
  return 0;
}
int hipMemGetInfo(size_t* f, size_t* total) {
  *f = freeBytes;
  *total = size_t(288) << 30;
  return 0;
}
int hipStreamBeginCapture(void*, int) {
  capture = new std::vector<Node>;
  return 0;
}
int hipStreamEndCapture(void*, void** graph) {
  *graph = capture;
  capture = nullptr;
  captures++;
  return 0;
}
int hipGraphInstantiate(void** exec, void* graph, void*, char*, size_t) {
  *exec = new std::vector<Node>(*static_cast<std::vector<Node>*>(graph));
  return 0;
}
int hipGraphLaunch(void* exec, void*) {
  for (const Node& n : *static_cast<std::vector<Node>*>(exec)) {
    bool ok = true;
    for (size_t i = 0; i < n.args.size(); i++)
      if (n.ids[i] >= 0 && !find(n.args[i])->live) {
        stale++;
        ok = false;
      }
    if (ok) effect(n);
  }
  return 0;
}
int hipGraphExecDestroy(void* exec) {
  delete static_cast<std::vector<Node>*>(exec);
  return 0;
}
int hipGraphDestroy(void* graph) {
  delete static_cast<std::vector<Node>*>(graph);
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
  static char region[4096];
  *p = region;
  return 0;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipGetLastError() { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  static int stream;
  *s = &stream;
  return 0;
}
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipEventCreate(void** e) {
  static int event;
  *e = &event;
  return 0;
}
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0;
  return 0;
}
int hipMemAddressReserve(void**, size_t, size_t, void*, unsigned long long) { return kUnsupported; }
int hipMemAddressFree(void*, size_t) { return kUnsupported; }
int hipMemCreate(void*, size_t, const void*, unsigned long long) { return kUnsupported; }
int hipMemRelease(void*) { return kUnsupported; }
int hipMemMap(void*, size_t, size_t, void*, unsigned long long) { return kUnsupported; }
int hipMemUnmap(void*, size_t) { return kUnsupported; }
int hipMemSetAccess(void*, size_t, const void*, size_t) { return kUnsupported; }
}
