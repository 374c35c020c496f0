// rt_xfer.hip -- a level's state between the host's doubles and the device.
//
// The host's arrays are ordinary memory, often fresh from the allocator.  A
// plain copy into them runs through the runtime's staging at 10.6 GB/s (the
// first touch of every page included), and the float fields need a conversion
// on top: reading 128^3 cells with three groups back took 28 ms that way,
// against 3.4 ms for their 193 MB over PCIe at the 57 GB/s that page-locked
// memory reaches.  So the arrays cross in their device type, in chunks through
// page-locked slots, and several host threads convert them (and take the page
// faults) side by side while the next chunks are in flight: 4.8 to 5.8 ms (5.5 ms
// for the way in, 22.5 before).  Up to a MiB of doubles, where the nine copies'
// latency is what counts, one kernel gathers all arrays, converted, straight into
// a slot (or scatters them from it).
#include <hip/hip_runtime.h>

#include <sched.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "rt_xfer.h"

namespace emma {
namespace {

// 128^3 cells with three groups (193 MB), both ways: chunks of 1 MiB 6.0 /
// 5.6 ms, of 512 KiB 6.8 / 6.5, of 256 KiB 8.8 / 8.6; of 2 MiB 5.6 / 4.8, but
// 64^3 cells with nine groups (55 MB) back then 1.7 instead of 1.45 ms and
// with one FP64 group (19 MB) 1.5 instead of 1.0 (fewer chunks than threads):
// 2 MiB from 128 MB on.  Twelve threads gain nothing over eight.
constexpr size_t kPackBytes = 1u << 20;  // up to here one gathering kernel
constexpr size_t kChunkBytes = 1u << 20, kLargeChunkBytes = 2u << 20, kLargeTotal = 128u << 20;
constexpr int kMaxThreads = 8;
constexpr size_t kBytesPerThread = 4u << 20;  // host bytes that pay for starting a thread (0.02 to 2 ms)
constexpr size_t kKeepBytes = 2 * kMaxThreads * kLargeChunkBytes;
constexpr size_t kIdleBytes = 2 * kMaxThreads * kChunkBytes;
constexpr size_t kKeepBlocks = 16;

// The page-locked memory of a transfer: one block, two slots of a chunk for each
// thread.  Freeing page-locked memory takes 0.28 ms a block whatever its size,
// and allocating 32 MiB 2.2 ms in one block, 6 in sixteen: closing the last
// context of a program after 64^3 cells and two finer levels, three FP64 groups,
// takes 5.8 ms, 9.7 with sixteen slots of their own, 4.8 with none.  The first
// touch of fresh ones costs 0.37 ms a MiB, so that a program of many short-lived
// contexts would pay more for its slots than they bring (32^3 cells, three FP64
// groups, a context made, set, read and closed: 1.45 ms, 2.95 with a new block):
// kIdleBytes stay with the process between contexts.
struct FreeBlock {
  char* p;
  size_t bytes;
};
std::mutex g_mu;
std::vector<FreeBlock> g_free;  // blocks nobody uses: kKeepBytes at most, kIdleBytes without a context
size_t g_kept = 0;
int g_users = 0;

// blocks taken off the list under the lock, freed after it
struct Gone {
  FreeBlock b[kKeepBlocks];
  size_t n = 0;
  void take(size_t i) {
    b[n++] = g_free[i];
    g_kept -= g_free[i].bytes;
    g_free.erase(g_free.begin() + i);
  }
  ~Gone() {
    for (size_t i = 0; i < n; i++) (void)hipHostFree(b[i].p);
  }
};

class Block {
 public:
  // n units of `unit` bytes, or the half, the quarter ... if there is no more
  Block(size_t n, size_t unit) {
    for (; n > 0 && p == nullptr; n /= 2) {
      take(n * unit);
      count = p != nullptr ? n : 0;
    }
  }
  ~Block() {
    if (p == nullptr) return;
    Gone gone;
    {
      std::lock_guard<std::mutex> lock(g_mu);
      const size_t keep = g_users > 0 ? kKeepBytes : kIdleBytes;
      if (bytes_ <= keep && g_free.capacity() >= kKeepBlocks) {
        while (g_kept + bytes_ > keep || g_free.size() >= kKeepBlocks) gone.take(0);
        g_free.push_back({p, bytes_});
        g_kept += bytes_;
        p = nullptr;
      }
    }
    if (p != nullptr) (void)hipHostFree(p);
  }
  Block(const Block&) = delete;
  Block& operator=(const Block&) = delete;

  char* p = nullptr;  // null: no page-locked memory to be had
  size_t count = 0;   // units

 private:
  void take(size_t want) {
    {
      std::lock_guard<std::mutex> lock(g_mu);
      size_t best = g_free.size();
      for (size_t i = 0; i < g_free.size(); i++)
        if (g_free[i].bytes >= want && (best == g_free.size() || g_free[i].bytes < g_free[best].bytes)) best = i;
      if (best < g_free.size()) {
        p = g_free[best].p;
        bytes_ = g_free[best].bytes;
        g_kept -= bytes_;
        g_free.erase(g_free.begin() + best);
        return;
      }
    }
    // coherent: a slot goes from kernel to host and back with no more than an
    // event in between (same rates either way, 50 GB/s in and 54 out)
    void* fresh = nullptr;
    if (hipHostMalloc(&fresh, want, hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess) {
      p = (char*)fresh;
      bytes_ = want;
    } else {
      (void)hipGetLastError();
    }
  }
  size_t bytes_ = 0;
};

// ---- a chunk of an array, and its conversion
struct Chunk {
  const XferPart* part;
  size_t first, n;
  size_t bytes() const { return n * (part->f32 ? sizeof(float) : sizeof(double)); }
  char* dev() const { return (char*)part->dev + first * (part->f32 ? sizeof(float) : sizeof(double)); }
};

void from_slot(const Chunk& c, const void* slot) {
  double* h = (double*)c.part->host + c.first;
  if (c.part->f32) {
    const float* f = (const float*)slot;
    for (size_t i = 0; i < c.n; i++) h[i] = (double)f[i];
  } else {
    memcpy(h, slot, c.n * sizeof(double));
  }
}

void into_slot(const Chunk& c, void* slot) {
  const double* h = (const double*)c.part->host + c.first;
  if (!c.part->f32) {
    memcpy(slot, h, c.n * sizeof(double));
    return;
  }
  float* f = (float*)slot;
  const double fl = c.part->floor;
  const float up = c.part->floor_up;
  if (fl > 0.) {
    for (size_t i = 0; i < c.n; i++) {
      const float v = (float)h[i];
      f[i] = (h[i] >= fl && (double)v < fl) ? up : v;
    }
  } else {
    for (size_t i = 0; i < c.n; i++) f[i] = (float)h[i];
  }
}

// ---- without page-locked memory: the runtime's copies, converted a piece at a time
template <bool ToHost>
hipError_t plain(hipStream_t s, const XferPart* parts, int np) {
  std::unique_ptr<char[]> piece(new (std::nothrow) char[kChunkBytes]);
  if (!piece) return hipErrorOutOfMemory;
  for (int k = 0; k < np; k++) {
    const size_t per = kChunkBytes / (parts[k].f32 ? sizeof(float) : sizeof(double));
    for (size_t i = 0; i < parts[k].n; i += per) {
      const Chunk c = {&parts[k], i, std::min(per, parts[k].n - i)};
      if (!ToHost) into_slot(c, piece.get());
      hipError_t e = ToHost ? hipMemcpyAsync(piece.get(), c.dev(), c.bytes(), hipMemcpyDeviceToHost, s)
                            : hipMemcpyAsync(c.dev(), piece.get(), c.bytes(), hipMemcpyHostToDevice, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e != hipSuccess) return e;
      if (ToHost) from_slot(c, piece.get());
    }
  }
  return hipSuccess;
}

// ---- one kernel for all arrays of a small level
struct PackArgs {
  int np;
  unsigned off[kMaxXferParts + 1];  // first element of each part
  XferPart part[kMaxXferParts];
};

template <bool ToHost>
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a, double* slot) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.off[a.np]) return;
  int k = 0;
  while (i >= a.off[k + 1]) k++;
  const XferPart& p = a.part[k];
  const unsigned j = i - a.off[k];
  if (ToHost) {
    slot[i] = p.f32 ? (double)((const float*)p.dev)[j] : ((const double*)p.dev)[j];
  } else {
    const double v = slot[i];
    if (p.f32) {
      float f = (float)v;
      if (v >= p.floor && (double)f < p.floor) f = p.floor_up;
      ((float*)p.dev)[j] = f;
    } else {
      ((double*)p.dev)[j] = v;
    }
  }
}

template <bool ToHost>
hipError_t packed(hipStream_t s, const XferPart* parts, int np, size_t total) {
  const Block slot(1, kPackBytes);
  if (slot.p == nullptr) return plain<ToHost>(s, parts, np);
  PackArgs a;
  a.np = np;
  a.off[0] = 0;
  for (int k = 0; k < np; k++) {
    a.part[k] = parts[k];
    a.off[k + 1] = a.off[k] + (unsigned)parts[k].n;
    if (!ToHost) memcpy((double*)slot.p + a.off[k], parts[k].host, parts[k].n * sizeof(double));
  }
  hipLaunchKernelGGL((pack_kernel<ToHost>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a, (double*)slot.p);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess && ToHost)
    for (int k = 0; k < np; k++) memcpy(parts[k].host, (double*)slot.p + a.off[k], parts[k].n * sizeof(double));
  return e;
}

// ---- chunks through slots
// A chunk's copy as a kernel, 16 bytes a thread: the runtime's copies cost
// about 35 us each on one stream whatever their size, kernels follow each
// other within a few (128^3 cells with three groups back, 1 MiB chunks: 6.9
// against 5.6 ms).
__global__ __launch_bounds__(256) void copy_kernel(uint4* dst, const uint4* src, unsigned n) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

hipError_t copy_chunk(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
  if (((size_t)dst | (size_t)src | bytes) & 15) return hipMemcpyAsync(dst, src, bytes, kind, s);
  const unsigned n = (unsigned)(bytes / 16);
  hipLaunchKernelGGL(copy_kernel, dim3((n + 255) / 256), dim3(256), 0, s, (uint4*)dst, (const uint4*)src, n);
  return hipGetLastError();
}

struct Job {
  int device;
  hipStream_t s;
  size_t chunk;  // bytes, at most
  const std::vector<Chunk>* chunks;
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
};

// one thread's share: two slots, one in flight while the other is converted
template <bool ToHost>
void work(Job& job, char* slots, bool own_thread) {
  auto failed = [&](hipError_t e) {
    if (e != hipSuccess) job.err = (int)e;
    return job.err != (int)hipSuccess;
  };
  if (own_thread && hipSetDevice(job.device) != hipSuccess) return;  // its chunks go to the others
  char* const slot[2] = {slots, slots + job.chunk};
  hipEvent_t ev[2] = {nullptr, nullptr};
  bool flying[2] = {false, false};
  for (auto& e : ev)
    if (failed(hipEventCreateWithFlags(&e, hipEventDisableTiming))) break;
  const std::vector<Chunk>& ch = *job.chunks;
  auto wait = [&](int b) {
    const hipError_t e = flying[b] ? hipEventSynchronize(ev[b]) : hipSuccess;
    flying[b] = false;
    return !failed(e);
  };
  auto send = [&](size_t k, int b) {
    const Chunk& c = ch[k];
    hipError_t e = ToHost ? copy_chunk(slot[b], c.dev(), c.bytes(), hipMemcpyDeviceToHost, job.s)
                          : copy_chunk(c.dev(), slot[b], c.bytes(), hipMemcpyHostToDevice, job.s);
    if (e == hipSuccess) {
      e = hipEventRecord(ev[b], job.s);
      flying[b] = e == hipSuccess;
    }
    return !failed(e);
  };
  int b = 0;
  if (job.err == (int)hipSuccess) {
    if (ToHost) {
      size_t k = job.next++;
      if (k < ch.size() && send(k, b)) {
        while (k < ch.size()) {
          const size_t n = job.next++;
          if (n < ch.size() && !send(n, 1 - b)) break;
          if (!wait(b)) break;
          from_slot(ch[k], slot[b]);
          k = n;
          b = 1 - b;
        }
      }
    } else {
      for (size_t k = job.next++; k < ch.size(); k = job.next++, b = 1 - b) {
        if (!wait(b)) break;
        into_slot(ch[k], slot[b]);
        if (!send(k, b)) break;
      }
    }
  }
  // no slot goes back while a copy may still use it
  for (int i = 0; i < 2; i++) (void)wait(i);
  if (job.err != (int)hipSuccess) (void)hipStreamSynchronize(job.s);
  for (auto e : ev)
    if (e) (void)hipEventDestroy(e);
}

int host_threads() {
  cpu_set_t set;
  CPU_ZERO(&set);
  const int n = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
  return std::max(1, std::min(kMaxThreads, n));
}

template <bool ToHost>
hipError_t chunked(int device, hipStream_t s, const XferPart* parts, int np, size_t total) {
  std::vector<Chunk> chunks;
  size_t moved = 0;
  for (int k = 0; k < np; k++) moved += parts[k].n * (parts[k].f32 ? sizeof(float) : sizeof(double));
  Job job;
  job.device = device;
  job.s = s;
  job.chunk = moved >= kLargeTotal ? kLargeChunkBytes : kChunkBytes;
  job.chunks = &chunks;
  for (int k = 0; k < np; k++) {
    const size_t per = job.chunk / (parts[k].f32 ? sizeof(float) : sizeof(double));
    for (size_t i = 0; i < parts[k].n; i += per) chunks.push_back({&parts[k], i, std::min(per, parts[k].n - i)});
  }
  const size_t bytes = total * sizeof(double);
  const size_t want = std::min<size_t>({(size_t)host_threads(), chunks.size(), 1 + bytes / kBytesPerThread});
  const Block slots(want, 2 * job.chunk);  // fewer slots, fewer threads
  if (slots.p == nullptr) return plain<ToHost>(s, parts, np);
  std::vector<std::thread> th;
  try {
    th.reserve(slots.count);
    for (size_t i = 1; i < slots.count; i++)
      th.emplace_back(work<ToHost>, std::ref(job), slots.p + 2 * i * job.chunk, true);
  } catch (...) {  // fewer threads: the ones that run take all chunks
  }
  work<ToHost>(job, slots.p, false);
  for (auto& t : th) t.join();
  return (hipError_t)job.err.load();
}

template <bool ToHost>
hipError_t transfer(int device, hipStream_t s, const XferPart* in, int nin) {
  const DeviceScope on(device);
  XferPart parts[kMaxXferParts];
  int np = 0;
  size_t total = 0;
  for (int k = 0; k < nin; k++) {
    if (in[k].n == 0) continue;
    if (np == kMaxXferParts) return hipErrorInvalidValue;
    parts[np++] = in[k];
    total += in[k].n;
  }
  if (np == 0) return hipStreamSynchronize(s);
  if (total * sizeof(double) <= kPackBytes) return packed<ToHost>(s, parts, np, total);
  try {
    return chunked<ToHost>(device, s, parts, np, total);
  } catch (...) {
    return hipErrorOutOfMemory;
  }
}

}  // namespace

hipError_t xfer_to_host(int device, hipStream_t s, const XferPart* parts, int np) {
  return transfer<true>(device, s, parts, np);
}
hipError_t xfer_to_device(int device, hipStream_t s, const XferPart* parts, int np) {
  return transfer<false>(device, s, parts, np);
}

void xfer_retain() {
  std::lock_guard<std::mutex> lock(g_mu);
  if (g_users++ > 0) return;
  // a device reset between contexts takes the blocks with it
  for (size_t i = g_free.size(); i-- > 0;) {
    unsigned flags = 0;
    if (hipHostGetFlags(&flags, g_free[i].p) == hipSuccess) continue;
    (void)hipGetLastError();
    g_kept -= g_free[i].bytes;
    g_free.erase(g_free.begin() + i);
  }
  try {
    g_free.reserve(kKeepBlocks);
  } catch (...) {  // nothing is kept then
  }
}

void xfer_release() {
  Gone gone;
  std::lock_guard<std::mutex> lock(g_mu);
  if (--g_users > 0) return;
  for (size_t i = g_free.size(); i-- > 0 && g_kept > kIdleBytes;)
    if (g_free[i].bytes > kIdleBytes) gone.take(i);
  while (g_kept > kIdleBytes) gone.take(0);
}

}  // namespace emma
