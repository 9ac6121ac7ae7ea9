// staging.hip -- copies between device memory and the caller's pageable buffers.
//
// HIP copies to pageable memory at 15-18 GB/s and from it at 21-31 GB/s on this
// machine (it pins or stages the caller's pages by itself), and a fresh buffer's
// first touch adds 12.6 ms per 256 MiB on one thread; a pinned copy runs at 50-57
// GB/s.  Here the data goes through pinned chunks: the DMA of later chunks overlaps
// the CPU's part (copy, first touch, and the conversion between FP32 psi and the
// caller's doubles), which large transfers spread over a few threads.
// Measured for psi downloads, before -> now: see copy_to_host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "ctx_internal.h"

namespace gpue {

namespace {

constexpr size_t CHUNK = (size_t)4 << 20;   // pinned bytes per buffer
constexpr int RING = 8;                     // buffers a transfer may hold
constexpr int POOLED = 16;                  // free buffers kept (64 MiB pinned), all devices together
constexpr int MAX_THREADS = 8;              // CPU threads of one large transfer
constexpr size_t MT_BYTES = (size_t)16 << 20;   // from here on a transfer uses threads
constexpr size_t DIRECT_UP = (size_t)8 << 20;   // smaller uploads: HIP's own path (66 us for 1 MiB, 148 for 4)

struct Buffer {
  void* p = nullptr;
  hipEvent_t ev = nullptr;   // the chunk's DMA
  int device = 0;
};

// Free buffers, shared by every context; given back to the system with the last one.
std::mutex pool_mu;
std::vector<Buffer> pool;
int users = 0;

void release(Buffer& b) {
  if (b.ev) (void)hipEventDestroy(b.ev);
  if (b.p) (void)hipHostFree(b.p);
  b = Buffer();
}

bool take(int device, Buffer& out) {
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    for (size_t k = 0; k < pool.size(); ++k)
      if (pool[k].device == device) {
        out = pool[k];
        pool.erase(pool.begin() + k);
        return true;
      }
  }
  Buffer b;
  b.device = device;
  if (hipHostMalloc(&b.p, CHUNK, hipHostMallocDefault) != hipSuccess ||
      hipEventCreateWithFlags(&b.ev, hipEventDisableTiming) != hipSuccess) {
    release(b);
    (void)hipGetLastError();
    return false;
  }
  out = b;
  return true;
}

// Whether the pool holds buffers for a transfer to overlap its halves.
bool pooled(int device) {
  std::lock_guard<std::mutex> lk(pool_mu);
  return std::count_if(pool.begin(), pool.end(), [&](const Buffer& b) { return b.device == device; }) >= 2;
}

void give(Buffer& b) {
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    if (users > 0 && pool.size() < (size_t)POOLED) {
      pool.push_back(b);
      return;
    }
  }
  release(b);
}

// One transfer: `n` elements of `es` bytes on the device; the caller's element has
// the same size, or is a double for a float (conv).
struct Job {
  char* host;
  char* dev;
  size_t n, es, per;   // elements, device bytes of one, elements per chunk
  bool conv, down;
  hipStream_t stream;
  int chunks, nbuf;
  Buffer buf[RING];
  std::atomic<int> next{0};          // next chunk for the CPU's part
  std::atomic<int> issued{0};        // chunks whose DMA is queued, in order
  std::atomic<int> filled[RING];     // upload: 1 + the chunk whose data a buffer holds; download: chunks consumed
  std::atomic<int> error{0};         // first hipError_t

  size_t count(int k) const { return std::min(per, n - (size_t)k * per); }
  void fail(hipError_t e) {
    int none = 0;
    error.compare_exchange_strong(none, (int)e);
  }
  void cpu_part(int k) {
    const size_t c = count(k), host_es = conv ? 8 : es;
    char* h = host + (size_t)k * per * host_es;
    void* b = buf[k % nbuf].p;
    if (!conv) {
      if (down) std::memcpy(h, b, c * es);
      else std::memcpy(b, h, c * es);
    } else if (down) {
      const float* f = (const float*)b;
      double* d = (double*)h;
      for (size_t i = 0; i < c; ++i) d[i] = f[i];
    } else {
      const double* d = (const double*)h;
      float* f = (float*)b;
      for (size_t i = 0; i < c; ++i) f[i] = (float)d[i];
    }
  }
  void queue(int k) {
    Buffer& b = buf[k % nbuf];
    const size_t bytes = count(k) * es;
    char* d = dev + (size_t)k * per * es;
    hipError_t e = down ? hipMemcpyAsync(b.p, d, bytes, hipMemcpyDeviceToHost, stream)
                        : hipMemcpyAsync(d, b.p, bytes, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess && chunks > 1) e = hipEventRecord(b.ev, stream);
    if (e != hipSuccess) fail(e);
    issued.store(k + 1, std::memory_order_release);
  }
  // Chunk k's DMA has ended.  A lone chunk is waited for with its stream: recording an
  // event and waiting for that takes 6-15 us more (us, event / stream: down 64 KiB 19.9 / 13.1,
  // 256 KiB 28.0 / 21.0, 1 MiB 69 / 62; 32 KiB FP32 down 19.6 / 12.4, up 30.2 / 14.4; HIP's own copies
  // from and to pageable memory take 12-22 us up to 256 KiB where they find the memory pinned
  // from the call before, and 50-190 where contexts of several sizes take turns).
  hipError_t wait(int k) { return chunks > 1 ? hipEventSynchronize(buf[k % nbuf].ev) : hipStreamSynchronize(stream); }
  // The CPU's part of chunks, as they come; every wait ends with the DMA of an
  // earlier chunk, with another thread's chunk, or with the error flag.
  void consume() {
    for (;;) {
      const int k = next.fetch_add(1);
      if (k >= chunks) return;
      const int need = down ? k + 1 : k - nbuf + 1;   // DMAs that must be queued before this part
      while (issued.load(std::memory_order_acquire) < need) {
        if (error.load()) return;
        std::this_thread::yield();
      }
      if (need > 0) {
        const hipError_t e = wait(k);
        if (e != hipSuccess) {
          fail(e);
          return;
        }
      }
      if (error.load()) return;
      cpu_part(k);
      filled[k % nbuf].store(k + 1, std::memory_order_release);
    }
  }
  // Queue the DMAs in order.  A download's chunk may take its buffer once the chunk
  // before it there is consumed, an upload's once the buffer is filled with it.
  // step(): as many as can go; true when all are queued, or after an error.
  bool step() {
    for (int k = issued.load(); k < chunks; k = issued.load()) {
      if (error.load()) return true;
      const int want = down ? k - nbuf + 1 : k + 1;
      if (want > 0 && filled[k % nbuf].load(std::memory_order_acquire) < want) return false;
      queue(k);
    }
    return true;
  }
};

// Without pinned memory to be had: HIP's own copies, conversions through a pageable chunk.
hipError_t run_pageable(const Job& j) {
  const size_t per = j.conv ? std::min(j.n, CHUNK / j.es) : j.n;
  std::unique_ptr<float[]> f;
  if (j.conv) {
    f.reset(new (std::nothrow) float[per]);
    if (!f) return hipErrorOutOfMemory;
  }
  for (size_t i = 0; i < j.n; i += per) {
    const size_t c = std::min(per, j.n - i);
    void* const dev = j.dev + i * j.es;
    double* const d = (double*)j.host + i;   // conv
    void* const host = j.conv ? (void*)f.get() : (void*)j.host;
    if (j.conv && !j.down)
      for (size_t k = 0; k < c; ++k) f[k] = (float)d[k];
    hipError_t e = j.down ? hipMemcpyAsync(host, dev, c * j.es, hipMemcpyDeviceToHost, j.stream)
                          : hipMemcpyAsync(dev, host, c * j.es, hipMemcpyHostToDevice, j.stream);
    if (e == hipSuccess) e = hipStreamSynchronize(j.stream);
    if (e != hipSuccess) return e;
    if (j.conv && j.down)
      for (size_t k = 0; k < c; ++k) d[k] = f[k];
  }
  return hipSuccess;
}

hipError_t run_on(Job& j, int device) {
  const size_t bytes = j.n * j.es;
  // one chunk up to 2 MiB, then chunks of 2 MiB up to 8 MiB: a chunk costs about 15 us
  // beside its bytes (256 KiB chunks: 90 us for 1 MiB down, 206 us for 4 MiB)
  const size_t chunk = bytes <= ((size_t)8 << 20) ? CHUNK / 2 : CHUNK;
  j.per = chunk / j.es;
  j.chunks = (int)((j.n + j.per - 1) / j.per);
  const int want = std::min(j.chunks, RING);
  for (j.nbuf = 0; j.nbuf < want && take(device, j.buf[j.nbuf]); ++j.nbuf) j.filled[j.nbuf] = 0;
  if (j.nbuf == 0) return run_pageable(j);
  std::vector<std::thread> th;
  if (bytes >= MT_BYTES) {
    const int hw = (int)std::thread::hardware_concurrency();
    const int nt = std::min(std::min(MAX_THREADS, j.chunks), std::max(1, hw / 2)) - 1;
    try {
      for (int t = 0; t < nt; ++t)
        th.emplace_back([&j, device] {
          (void)hipSetDevice(device);
          j.consume();
        });
    } catch (const std::exception&) {
      // fewer threads: the loop below takes every chunk nobody else takes
    }
  }
  if (th.empty()) {
    // one thread: queue what can go, then the next chunk's CPU part
    while (!j.error.load() && j.next.load() < j.chunks) {
      (void)j.step();
      const int k = j.next.load();
      if (j.error.load()) break;
      if (j.down || k >= j.nbuf) {
        const hipError_t e = j.wait(k);
        if (e != hipSuccess) {
          j.fail(e);
          break;
        }
      }
      j.cpu_part(k);
      j.filled[k % j.nbuf] = k + 1;
      j.next = k + 1;
    }
    if (!j.error.load()) (void)j.step();
  } else {
    while (!j.step()) std::this_thread::yield();
    if (j.down) j.consume();
  }
  for (std::thread& t : th) t.join();
  // an upload ends with its last DMAs; after an error nothing may still use the buffers
  if (!j.down || j.error.load())
    for (int b = 0; b < j.nbuf; ++b)
      if (j.issued.load() > b) {
        const hipError_t e = j.wait(b);
        if (e != hipSuccess) j.fail(e);
      }
  for (int b = 0; b < j.nbuf; ++b) give(j.buf[b]);
  return (hipError_t)j.error.load();
}

// On the stream's device: the buffers' events belong to it.
hipError_t run(Job& j, int device) {
  if (j.n == 0) return hipSuccess;
  int cur = device;
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != device) e = hipSetDevice(device);
  if (e == hipSuccess) e = run_on(j, device);
  if (cur != device) (void)hipSetDevice(cur);
  return e;
}

}  // namespace

void staging_acquire() {
  std::lock_guard<std::mutex> lk(pool_mu);
  ++users;
}

void staging_release() {
  std::vector<Buffer> old;
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    if (--users > 0) return;
    old.swap(pool);
  }
  for (Buffer& b : old) release(b);
}

// n elements of es bytes from dev (work on `stream` first) to the caller's buffer, or
// floats to doubles (widen); returns when they are there.  Median of a psi download
// into a new numpy array, before -> now: 64 MiB 6.3 -> 2.0 ms, 256 MiB 25.5 -> 6.4 ms,
// 256^3 FP32 (128 MiB to 256) 48.1 -> 5.2 ms.
hipError_t copy_to_host(void* host, const void* dev, size_t n, size_t es, bool widen, int device,
                        hipStream_t stream) {
  Job j;
  j.host = (char*)host;
  j.dev = (char*)const_cast<void*>(dev);
  j.n = n;
  j.es = es;
  j.conv = widen;
  j.down = true;
  j.stream = stream;
  return run(j, device);
}

// The other way (doubles rounded to floats with `narrow`); returns when the device
// holds them.  64 MiB 2.3 -> 1.7 ms, 256 MiB 8.9 -> 5.9 ms, 256^3 FP32 38.1 -> 3.5 ms.
// A program's first upload, without conversion, takes HIP's own path too: allocating the
// ring (about 0.4 ms a buffer) would cost more than it saves (a new 128 x 128 x 96
// context with its upload took 12.8 ms, with the ring 15.4).
hipError_t copy_to_device(void* dev, const void* host, size_t n, size_t es, bool narrow, int device,
                          hipStream_t stream) {
  Job j;
  j.host = (char*)const_cast<void*>(host);
  j.dev = (char*)dev;
  j.n = n;
  j.es = es;
  j.conv = narrow;
  j.down = false;
  j.stream = stream;
  if (!narrow && (n * es < DIRECT_UP || !pooled(device))) {
    hipError_t e = hipMemcpyAsync(dev, host, n * es, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    return e;
  }
  return run(j, device);
}

}  // namespace gpue
