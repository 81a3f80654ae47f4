// Large copies between the device and pageable host memory, through pinned
// chunks and several threads.
//
// hipMemcpyAsync on pageable memory moves 16 GB/s into pages it has pinned
// before and a third of that into fresh ones.  Here each thread moves every
// so-many-th chunk -- by DMA to or from its own pinned chunk, by memcpy to or
// from the caller's memory -- so that first touches and copies of several
// chunks overlap the DMA of others: 23 MB into a warm array 1.4 ms -> 0.70, a
// wired network of 190 MB and its export 29.3 -> 11.6, a checkpoint of 18 MB
// saved and restored 4.1 -> 2.6.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#include "nc_internal.h"

namespace nc {
namespace {

// A chunk costs about 20 us beside its DMA: 23 MB in chunks of 256 KiB 1.7 ms,
// 512 KiB 1.15, 1 MiB 0.82, 2 MiB 0.70, whatever the threads from four on.
constexpr size_t kChunk = 2u << 20;
constexpr unsigned kThreads = 4;
// Pinned buffers and streams kept between calls: while simulations live (a
// server builds on four threads), and for programs that only wire networks.
constexpr size_t kIdleMost = 6, kIdleAlone = 1;

struct PinnedChunks {
  int device = 0;
  unsigned char* p = nullptr;  // kThreads chunks
  hipEvent_t ev[kThreads] = {};
  ~PinnedChunks() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (p) (void)hipHostFree(p);
  }
};

// Idle things of a device each, no allocation to keep one.
template <class T>
struct Idle {
  struct Item {
    int device;
    T x;
  } item[kIdleMost] = {};
  size_t n = 0;
  bool take(int device, T* out) {
    for (size_t i = 0; i < n; ++i)
      if (item[i].device == device) {
        *out = item[i].x;
        item[i] = item[--n];
        return true;
      }
    return false;
  }
  bool give(int device, T x, size_t most) {
    if (n >= most) return false;
    item[n++] = Item{device, x};
    return true;
  }
};

std::mutex g_mu;
Idle<PinnedChunks*> g_idle;
Idle<hipStream_t> g_streams;
unsigned g_users = 0;  // simulations alive
size_t idle_most() { return g_users ? kIdleMost : kIdleAlone; }

hipError_t take(int device, PinnedChunks** out) {
  {
    std::lock_guard<std::mutex> g(g_mu);
    if (g_idle.take(device, out)) return hipSuccess;
  }
  PinnedChunks* b = new PinnedChunks();
  b->device = device;
  hipError_t e = hipHostMalloc((void**)&b->p, kThreads * kChunk, hipHostMallocDefault);
  for (unsigned t = 0; t < kThreads && e == hipSuccess; ++t)
    e = hipEventCreateWithFlags(&b->ev[t], hipEventDisableTiming);
  if (e != hipSuccess) {
    delete b;
    return e;
  }
  *out = b;
  return hipSuccess;
}

void give_back(PinnedChunks* b) {
  {
    std::lock_guard<std::mutex> g(g_mu);
    if (g_idle.give(b->device, b, idle_most())) return;
  }
  delete b;
}

// Without a pinned buffer.
hipError_t move_direct(hipStream_t st, const Segment* seg, size_t n_seg, bool to_host) {
  hipError_t e = hipSuccess;
  for (size_t i = 0; i < n_seg && e == hipSuccess; ++i)
    if (seg[i].bytes)
      e = to_host ? hipMemcpyAsync(seg[i].host, seg[i].dev, seg[i].bytes, hipMemcpyDeviceToHost, st)
                  : hipMemcpyAsync(seg[i].dev, seg[i].host, seg[i].bytes, hipMemcpyHostToDevice, st);
  const hipError_t w = hipStreamSynchronize(st);
  return e == hipSuccess ? w : e;
}

hipError_t move(int device, hipStream_t st, const Segment* seg, size_t n_seg, bool to_host) {
  std::vector<Segment> chunks;
  for (size_t i = 0; i < n_seg; ++i)
    for (size_t a = 0; a < seg[i].bytes; a += kChunk)
      chunks.push_back(Segment{(char*)seg[i].host + a, (char*)seg[i].dev + a, std::min(kChunk, seg[i].bytes - a)});
  if (chunks.empty()) return hipSuccess;
  size_t total = 0;
  for (const Segment& c : chunks) total += c.bytes;
  std::vector<std::thread> th;
  th.reserve(kThreads);
  PinnedChunks* b = nullptr;
  hipError_t e = take(device, &b);
  if (e != hipSuccess) {
    // the host has no more memory to pin, which the copies themselves can do
    // without
    (void)hipGetLastError();
    return move_direct(st, seg, n_seg, to_host);
  }
  if (total <= kChunk) {
    // one wait for all of it
    size_t at = 0;
    for (const Segment& c : chunks) {
      if (!to_host) memcpy(b->p + at, c.host, c.bytes);
      if (e == hipSuccess)
        e = to_host ? hipMemcpyAsync(b->p + at, c.dev, c.bytes, hipMemcpyDeviceToHost, st)
                    : hipMemcpyAsync(c.dev, b->p + at, c.bytes, hipMemcpyHostToDevice, st);
      at += c.bytes;
    }
    const hipError_t w = hipStreamSynchronize(st);
    if (e == hipSuccess) e = w;
    at = 0;
    for (const Segment& c : chunks) {
      if (to_host && e == hipSuccess) memcpy(c.host, b->p + at, c.bytes);
      at += c.bytes;
    }
    give_back(b);
    return e;
  }
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  auto work = [&](unsigned t) {
    hipError_t x = hipSetDevice(device);
    unsigned char* const pin = b->p + t * kChunk;
    while (x == hipSuccess && err.load() == (int)hipSuccess) {
      const size_t i = next.fetch_add(1);
      if (i >= chunks.size()) return;
      const Segment& c = chunks[i];
      if (to_host) x = hipMemcpyAsync(pin, c.dev, c.bytes, hipMemcpyDeviceToHost, st);
      else {
        memcpy(pin, c.host, c.bytes);
        x = hipMemcpyAsync(c.dev, pin, c.bytes, hipMemcpyHostToDevice, st);
      }
      if (x == hipSuccess) x = hipEventRecord(b->ev[t], st);
      if (x == hipSuccess) x = hipEventSynchronize(b->ev[t]);
      if (x == hipSuccess && to_host) memcpy(c.host, pin, c.bytes);
    }
    if (x != hipSuccess) err.store((int)x);
  };
  const unsigned nt = (unsigned)std::min<size_t>(
      {chunks.size(), kThreads, std::max<size_t>(1, std::thread::hardware_concurrency())});
  try {
    for (unsigned t = 1; t < nt; ++t) th.emplace_back(work, t);
  } catch (const std::exception&) {
    // no thread, or no memory for one, to be had: the others move all chunks
    // (those started have to be joined whatever it was)
  }
  work(0);
  for (auto& t : th) t.join();
  if (err.load() != (int)hipSuccess) (void)hipStreamSynchronize(st);  // nothing may still use the pinned chunks
  give_back(b);
  return (hipError_t)err.load();
}

}  // namespace

hipError_t download(int device, hipStream_t st, const Segment* seg, size_t n_seg) {
  return move(device, st, seg, n_seg, true);
}
hipError_t upload(int device, hipStream_t st, const Segment* seg, size_t n_seg) {
  return move(device, st, seg, n_seg, false);
}

hipError_t stream_take(int device, hipStream_t* out) {
  {
    std::lock_guard<std::mutex> g(g_mu);
    if (g_streams.take(device, out)) return hipSuccess;
  }
  return hipStreamCreateWithFlags(out, hipStreamNonBlocking);
}

void stream_give(int device, hipStream_t st) {
  (void)hipStreamSynchronize(st);
  {
    std::lock_guard<std::mutex> g(g_mu);
    if (g_streams.give(device, st, idle_most())) return;
  }
  (void)hipStreamDestroy(st);
}

void xfer_user(int change) {
  Idle<PinnedChunks*> gone;
  Idle<hipStream_t> streams;
  {
    std::lock_guard<std::mutex> g(g_mu);
    g_users += (unsigned)change;
    if (g_users == 0) {
      std::swap(gone, g_idle);
      std::swap(streams, g_streams);
    }
  }
  for (size_t i = 0; i < gone.n; ++i) delete gone.item[i].x;
  for (size_t i = 0; i < streams.n; ++i) (void)hipStreamDestroy(streams.item[i].x);
}

}  // namespace nc
