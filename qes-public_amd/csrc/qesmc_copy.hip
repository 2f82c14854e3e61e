// Large copies between the caller's (pageable) arrays and the device.
//
// The runtime's own copy to pageable memory moves about 11 GB/s where the
// array's pages are touched for the first time (one thread faults them in and
// copies from a staging buffer), against 57 GB/s for the link with pinned
// memory: u, v, w of a 1000 x 1000 x 150 city took 171 ms.  Here the caller
// queues the copies of successive chunks through a ring of pinned slots on one
// stream, and worker threads move each slot to or from the array as its turn
// comes, so the link, the page faults and the host copies overlap.
//
// Memory that the runtime knows (pinned, managed, another device array) it
// copies itself, at the link's rate: u, v, w of 400 x 400 x 120 cells into pinned
// arrays take 4.15 ms so and 5.30 through the slots.
//
// The slots belong to the process: one set per device, made once the large
// copies since they were last freed amount to 64 MiB (making and freeing them takes
// 3.6 ms, which 13 MB of a context that then goes do not repay: set-up, run, copy and
// close of 128 x 128 x 64 cells took 5.2 ms without them and 9.1 with), lent to one call at a time (a call that finds it lent takes the
// runtime's copy) and freed with the device's last context.
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "qesmc_internal.h"

namespace {

constexpr int kWorkers = 8;
constexpr int kSlots = 12;
constexpr size_t kSlotBytes = (size_t)4 << 20;
constexpr size_t kLeastChunk = (size_t)1 << 20;
// Below these the threads cost more than they save: towards the host 6.4 MB
// take 0.34 ms either way; towards the device the runtime's copy, which has no
// pages to fault in, reaches 31 GB/s.
constexpr size_t kLeastToHost = (size_t)8 << 20;
constexpr size_t kLeastToDevice = (size_t)128 << 20;
constexpr size_t kRepay = (size_t)64 << 20;
constexpr int kMaxDevices = 64;

struct Slots {
  std::mutex mu;
  int contexts = 0;
  bool lent = false;
  size_t without = 0;  // bytes of large copies made without the slots, while there are none
  void *pinned[kSlots] = {};
  hipEvent_t done[kSlots] = {};  // the slot's last copy over the link
  hipStream_t stream = nullptr;
};

Slots g_slots[kMaxDevices];

void free_slots(Slots &s)
{
  for (int q = 0; q < kSlots; ++q) {
    if (s.done[q]) (void)hipEventDestroy(s.done[q]);
    if (s.pinned[q]) (void)hipHostFree(s.pinned[q]);
    s.done[q] = nullptr;
    s.pinned[q] = nullptr;
  }
  if (s.stream) (void)hipStreamDestroy(s.stream);
  s.stream = nullptr;
  s.without = 0;
}

// The device's slots for a copy of `bytes`, made if need be; false if they are
// lent, do not repay yet or cannot be had.
bool borrow(Slots &s, size_t bytes)
{
  std::lock_guard<std::mutex> lock(s.mu);
  if (s.lent) return false;
  if (!s.stream && (s.without += bytes) < kRepay) return false;
  bool ok = s.stream || hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) == hipSuccess;
  for (int q = 0; q < kSlots && ok; ++q) {
    ok = (s.pinned[q] || hipHostMalloc(&s.pinned[q], kSlotBytes, hipHostMallocDefault) == hipSuccess) &&
         (s.done[q] || hipEventCreateWithFlags(&s.done[q], hipEventDisableTiming) == hipSuccess);
  }
  if (!ok) {
    (void)hipGetLastError();
    free_slots(s);
    return false;
  }
  s.lent = true;
  return true;
}

void give_back(Slots &s)
{
  std::lock_guard<std::mutex> lock(s.mu);
  s.lent = false;
}

// Whether the runtime has this memory on its books, or a worker may touch it.
bool known(const void *p)
{
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

hipError_t queue(hipStream_t st, const qesmc::HostPiece &p, bool to_device)
{
  if (p.bytes == 0) return hipSuccess;
  return to_device ? hipMemcpyAsync(p.device, p.host, p.bytes, hipMemcpyHostToDevice, st)
                   : hipMemcpyAsync(p.host, p.device, p.bytes, hipMemcpyDeviceToHost, st);
}

hipError_t plain(hipStream_t st, const qesmc::HostPiece *p, int n, bool to_device)
{
  for (int q = 0; q < n; ++q) {
    const hipError_t e = queue(st, p[q], to_device);
    if (e != hipSuccess) return e;
  }
  return hipStreamSynchronize(st);
}

}  // namespace

namespace qesmc {

void host_copy_attach(int device)
{
  if (device < 0 || device >= kMaxDevices) return;
  std::lock_guard<std::mutex> lock(g_slots[device].mu);
  ++g_slots[device].contexts;
}

void host_copy_detach(int device)
{
  if (device < 0 || device >= kMaxDevices) return;
  Slots &s = g_slots[device];
  std::lock_guard<std::mutex> lock(s.mu);
  if (--s.contexts == 0 && !s.lent) free_slots(s);
}

// Copy every piece, after all earlier work of `st` on `device` (the current
// device); returns when the copies are complete.
hipError_t host_copy(int device, hipStream_t st, const HostPiece *p, int n, bool to_device)
{
  const size_t least = to_device ? kLeastToDevice : kLeastToHost;
  size_t total = 0;
  for (int q = 0; q < n; ++q) total += p[q].bytes;
  if (total >= least)
    for (int q = 0; q < n; ++q)
      if (known(p[q].host)) total -= p[q].bytes;
  if (total < least || device < 0 || device >= kMaxDevices) return plain(st, p, n, to_device);
  size_t chunk = total / (2 * kSlots);
  chunk = chunk < kLeastChunk ? kLeastChunk : chunk > kSlotBytes ? kSlotBytes : chunk;
  struct Chunk {
    char *host, *device;
    size_t bytes;
  };
  std::vector<Chunk> chunks;
  std::vector<std::atomic<int>> state;  // 0 untouched, 1 in the slot or on its way, 2 finished
  try {
    for (int q = 0; q < n; ++q) {
      if (known(p[q].host)) continue;
      for (size_t o = 0; o < p[q].bytes; o += chunk)
        chunks.push_back({(char *)p[q].host + o, (char *)p[q].device + o,
                          p[q].bytes - o < chunk ? p[q].bytes - o : chunk});
    }
    state = std::vector<std::atomic<int>>(chunks.size());
  } catch (const std::bad_alloc &) {
    return plain(st, p, n, to_device);
  }
  Slots &s = g_slots[device];
  if (!borrow(s, total)) return plain(st, p, n, to_device);
  hipError_t first = hipSuccess;
  for (int q = 0; q < n && first == hipSuccess; ++q)
    if (known(p[q].host)) first = queue(st, p[q], to_device);
  const hipError_t waited = hipStreamSynchronize(st);
  if (first == hipSuccess) first = waited;
  if (first == hipSuccess) {
    const size_t count = chunks.size();
    std::atomic<size_t> next{0};
    std::atomic<bool> stop{false};
    std::atomic<int> failed{(int)hipSuccess};
    auto fail = [&](hipError_t e) {
      failed = (int)e;
      stop = true;
    };
    // a state another thread will set
    auto await = [&](size_t c, int value) {
      for (int spins = 0; state[c].load(std::memory_order_acquire) < value; ++spins) {
        if (stop) return false;
        if (spins > 200) std::this_thread::yield();
      }
      return true;
    };
    // slot c % kSlots: a worker moves chunk c between it and the array
    auto work = [&]() {
      if (hipSetDevice(device) != hipSuccess) return fail(hipErrorInvalidDevice);
      for (;;) {
        const size_t c = next.fetch_add(1);
        if (c >= count || stop) return;
        const int q = (int)(c % kSlots);
        if (to_device) {
          // the slot is free once chunk c - kSlots is across
          if (c >= (size_t)kSlots) {
            if (!await(c - kSlots, 2)) return;
            const hipError_t e = hipEventSynchronize(s.done[q]);
            if (e != hipSuccess) return fail(e);
          }
          std::memcpy(s.pinned[q], chunks[c].host, chunks[c].bytes);
          state[c].store(1, std::memory_order_release);
        } else {
          if (!await(c, 1)) return;
          const hipError_t e = hipEventSynchronize(s.done[q]);
          if (e != hipSuccess) return fail(e);
          std::memcpy(chunks[c].host, s.pinned[q], chunks[c].bytes);
          state[c].store(2, std::memory_order_release);
        }
      }
    };
    std::thread threads[kWorkers];
    int started = 0;
    const int want = (int)(count / 2 < (size_t)kWorkers ? count / 2 : (size_t)kWorkers);
    try {
      for (; started < want; ++started) threads[started] = std::thread(work);
    } catch (const std::exception &) {
      // no thread or no memory for one: fewer do the work; without any the runtime does
    }
    if (started == 0) {
      give_back(s);
      return plain(st, p, n, to_device);
    }
    // the caller queues the chunks in order
    for (size_t c = 0; c < count && !stop; ++c) {
      const int q = (int)(c % kSlots);
      hipError_t e;
      if (to_device) {
        if (!await(c, 1)) break;
        e = hipMemcpyAsync(chunks[c].device, s.pinned[q], chunks[c].bytes, hipMemcpyHostToDevice, s.stream);
        if (e == hipSuccess) e = hipEventRecord(s.done[q], s.stream);
        state[c].store(2, std::memory_order_release);
      } else {
        if (c >= (size_t)kSlots && !await(c - kSlots, 2)) break;
        e = hipMemcpyAsync(s.pinned[q], chunks[c].device, chunks[c].bytes, hipMemcpyDeviceToHost, s.stream);
        if (e == hipSuccess) e = hipEventRecord(s.done[q], s.stream);
        state[c].store(1, std::memory_order_release);
      }
      if (e != hipSuccess) fail(e);
    }
    for (int w = 0; w < started; ++w) threads[w].join();
    first = hipStreamSynchronize(s.stream);
    if (failed.load() != (int)hipSuccess) first = (hipError_t)failed.load();
  }
  give_back(s);
  return first;
}

}  // namespace qesmc
