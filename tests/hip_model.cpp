// hip_model.cpp -- a host model of the HIP runtime calls libemma_rt.so makes,
// for tests of its host code without a GPU.  Loaded with RTLD_GLOBAL before
// the library, so that the library's calls bind to it.  Two devices; device
// memory is host memory; streams run at once.  Kernels are not run, except the
// few that the host code waits for or whose data it reads back: copies, and
// the report of a call's end.
//
// What it holds the caller to: an event and the stream it is recorded on
// belong to one device; memory is freed once; a captured side stream is joined
// before the capture ends, and is of no use until it is destroyed otherwise.
// model_set() makes calls fail; the model_ functions report what was called.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include <time.h>

namespace {

struct Block {
  size_t bytes;
  unsigned flags;
  bool host;
};
std::recursive_mutex mu;
std::map<char*, Block> blocks;     // allocations, and ranges given with model_lock
std::map<const void*, std::string> kernels;
std::map<const void*, void*> symbols;
std::string launched;              // names of the kernels launched, in order
thread_local int device = 0;
thread_local std::vector<char> pushed;
thread_local hipError_t last = hipSuccess;  // of the launches

struct Stream {
  int device;
  int capture = 0;  // 1 the capturing stream, 2 a side stream drawn into it, 3 left unjoined
  std::vector<void*> records;  // call-end reports among the captured launches
  Stream* origin = nullptr;
};
struct Event {
  int device;
  Stream* on = nullptr;
};
std::vector<Stream*> streams;

std::string meanwhile_name;
void (*meanwhile)() = nullptr;

enum Key { kFailLaunch, kHostBytes, kDelayFlag, kCount };
long keys[kCount] = {-1, -1, 0};
std::atomic<int> pending{0};       // reports on their way
long host_blocks = 0, host_bytes = 0, host_allocs = 0, stream_waits = 0, cleared = 0;

Block* block_of(const void* p, char** base) {
  auto it = blocks.upper_bound((char*)p);
  if (it == blocks.begin()) return nullptr;
  --it;
  if ((char*)p >= it->first + it->second.bytes) return nullptr;
  *base = it->first;
  return &it->second;
}

hipError_t alloc(void** p, size_t n, unsigned flags, bool host) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (host && keys[kHostBytes] >= 0 && host_bytes + (long)n > keys[kHostBytes]) return hipErrorOutOfMemory;
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  memset(*p, 0, n);
  blocks[(char*)*p] = {n, flags, host};
  if (host) {
    host_blocks++;
    host_allocs++;
    host_bytes += n;
  }
  return hipSuccess;
}

hipError_t release(void* p, bool host) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  if (p == nullptr) return hipSuccess;
  auto it = blocks.find((char*)p);
  if (it == blocks.end() || it->second.host != host) return hipErrorInvalidValue;
  if (host) {
    host_blocks--;
    host_bytes -= it->second.bytes;
  }
  blocks.erase(it);
  free(p);
  return hipSuccess;
}

struct Record {  // CallRecord of rt_kernels.h
  int status[3];
  int flag;
  unsigned long long counts[3];
};

void report(void* rec) {
  auto set = [rec] {
    memset(((Record*)rec)->status, 0, 3 * sizeof(int));
    __atomic_store_n(&((Record*)rec)->flag, 1, __ATOMIC_RELEASE);
  };
  if (keys[kDelayFlag] == 0) return set();
  pending++;
  std::thread([set] {  // a worker that needs its share of a core for it
    timespec t;
    do {
      clock_gettime(CLOCK_THREAD_CPUTIME_ID, &t);
    } while (t.tv_sec * 1000000L + t.tv_nsec / 1000 < keys[kDelayFlag]);
    set();
    pending--;
  }).detach();
}

bool unusable(Stream* s) { return s != nullptr && s->capture == 3; }

}  // namespace

extern "C" {

// ---- the tests' side
void model_set(int key, long value) { keys[key] = value; }
long model_host_blocks() { return host_blocks; }
long model_host_bytes() { return host_bytes; }
long model_host_allocs() { return host_allocs; }
long model_stream_waits() { return stream_waits; }
long model_cleared() { return cleared; }  // list lengths the last call's end cleared
void model_device(int d) { device = d; }
int model_current() { return device; }
const char* model_launched() { return launched.c_str(); }
void model_forget() { launched.clear(); }
// what a device reset does: no block is known any more
void model_reset() {
  blocks.clear();
  host_blocks = host_bytes = 0;
}
// called when a kernel of that name is launched: what another thread does meanwhile
void model_during(const char* name, void (*f)()) {
  meanwhile_name = name;
  meanwhile = f;
}
// the flags that all page-locked blocks have in common
unsigned model_common_flags() {
  unsigned f = ~0u;
  for (auto& b : blocks)
    if (b.second.host) f &= b.second.flags;
  return f;
}
// ordinary memory the caller locked himself, as hipHostRegister would
void model_lock(void* p, size_t n, unsigned flags) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  blocks[(char*)p] = {n, flags, true};
}

// ---- devices and errors
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
hipError_t hipSetDevice(int d) { return device = d, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  return last = hipSuccess, e;
}
const char* hipGetErrorString(hipError_t) { return "model"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 4, hipSuccess; }

// ---- memory
hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n, 0, false); }
hipError_t hipFree(void* p) { return release(p, false); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) { return alloc(p, n, flags, true); }
hipError_t hipHostFree(void* p) { return release(p, true); }
hipError_t hipMemset(void* p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipHostGetFlags(unsigned* flags, void* p) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  char* base;
  Block* b = block_of(p, &base);
  if (b == nullptr || !b->host) return hipErrorInvalidValue;
  return *flags = b->flags, hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* at, size_t* n, hipDeviceptr_t p) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  char* base;
  Block* b = block_of(p, &base);
  if (b == nullptr) return hipErrorNotFound;
  return *at = base, *n = b->bytes, hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  char* base;
  Block* b = block_of(p, &base);
  memset(a, 0, sizeof(*a));
  a->type = b == nullptr ? hipMemoryTypeUnregistered : b->host ? hipMemoryTypeHost : hipMemoryTypeDevice;
  if (b != nullptr) {
    a->devicePointer = a->hostPointer = (void*)p;
    a->allocationFlags = b->flags;
  }
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
  auto it = symbols.find(symbol);
  if (it == symbols.end()) return hipErrorInvalidSymbol;
  return *p = it->second, hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreate(hipStream_t* s) {
  Stream* n = new Stream{device};
  streams.push_back(n);
  return *s = (hipStream_t)n, hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  for (auto& p : streams)
    if (p == (Stream*)s) p = nullptr;
  return delete (Stream*)s, hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  stream_waits++;
  if (unusable((Stream*)s)) return hipErrorStreamCaptureInvalidated;
  while (pending > 0) std::this_thread::sleep_for(std::chrono::microseconds(50));
  return hipSuccess;
}
static hipError_t event(hipEvent_t* e) { return *e = (hipEvent_t) new Event{device}, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return event(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return event(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (Event*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (unusable((Stream*)s)) return hipErrorStreamCaptureInvalidated;
  if (((Event*)e)->device != ((Stream*)s)->device) return hipErrorInvalidHandle;
  return ((Event*)e)->on = (Stream*)s, hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  Stream *to = (Stream*)s, *from = ((Event*)e)->on;
  if (unusable(to)) return hipErrorStreamCaptureInvalidated;
  if (from == nullptr) return hipSuccess;
  if (from->capture == 1 && to != from) {
    to->capture = 2;
    to->origin = from;
  } else if (from->capture == 2 && to == from->origin) {
    from->capture = 0;
  }
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  ((Stream*)s)->capture = 1;
  ((Stream*)s)->records.clear();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  Stream* st = (Stream*)s;
  st->capture = 0;
  bool unjoined = false;
  for (Stream* p : streams)
    if (p != nullptr && p->capture == 2 && p->origin == st) {
      p->capture = 3;
      unjoined = true;
    }
  if (unjoined) return hipErrorStreamCaptureUnjoined;
  return *g = (hipGraph_t) new std::vector<void*>(st->records), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete (std::vector<void*>*)g, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  return *x = (hipGraphExec_t) new std::vector<void*>(*(std::vector<void*>*)g), hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return delete (std::vector<void*>*)x, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
  for (void* r : *(std::vector<void*>*)x) report(r);
  return hipSuccess;
}

// ---- kernels
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t n, int, int) { symbols[var] = calloc(1, n); }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
  pushed.resize(sizeof(grid) + sizeof(block) + sizeof(shared) + sizeof(s));
  char* p = pushed.data();
  memcpy(p, &grid, sizeof(grid));
  memcpy(p + sizeof(grid), &block, sizeof(block));
  memcpy(p + sizeof(grid) + sizeof(block), &shared, sizeof(shared));
  memcpy(p + sizeof(grid) + sizeof(block) + sizeof(shared), &s, sizeof(s));
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
  const char* p = pushed.data();
  memcpy(grid, p, sizeof(*grid));
  memcpy(block, p + sizeof(*grid), sizeof(*block));
  memcpy(shared, p + sizeof(*grid) + sizeof(*block), sizeof(*shared));
  memcpy(s, p + sizeof(*grid) + sizeof(*block) + sizeof(*shared), sizeof(*s));
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lock(mu);
  Stream* st = (Stream*)s;
  if (unusable(st)) return last = hipErrorStreamCaptureInvalidated;
  const std::string& name = kernels[f];
  if (keys[kFailLaunch] >= 0 && keys[kFailLaunch]-- == 0) return last = hipErrorLaunchFailure;
  launched += name + "\n";
  if (meanwhile != nullptr && name.find(meanwhile_name) != std::string::npos) meanwhile();
  if (name.find("copy_kernel") != std::string::npos) {
    memcpy(*(void**)args[0], *(void**)args[1], (size_t) * (unsigned*)args[2] * 16);
  } else if (name.find("call_end_kernel") != std::string::npos) {
    cleared = *(int*)args[3];
    if (st->capture != 0)
      st->records.push_back(*(void**)args[4]);
    else
      report(*(void**)args[4]);
  }
  return hipSuccess;
}

}  // extern "C"
