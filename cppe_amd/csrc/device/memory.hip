// Chunk pool, arenas and pinned staging (memory.hh).
#include "memory.hh"

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

namespace cppe_dev {

// Largest allocation that succeeds: a bound for tests of what happens when there is no memory.
static std::atomic<size_t> g_most{SIZE_MAX};
extern "C" void cppe_hip_test_largest_allocation(long long bytes) {
  g_most = bytes > 0 ? (size_t)bytes : SIZE_MAX;
}

// ---- chunks ----------------------------------------------------------------------------------
// A chunk is at least kChunkMin and grows with what the arena holds already, so a system of any size has
// few and a small one (some ten blocks of 64 KiB and more at 1,000 sites) holds little; a request above
// kChunkPooled has a chunk of its own, which goes back to the device when it is free.
constexpr size_t kChunkMin    = size_t(2) << 20;
constexpr size_t kChunkPooled = size_t(256) << 20;
constexpr size_t kPoolBytes   = size_t(512) << 20;  // most the pool holds over all devices
constexpr auto kPoolAge       = std::chrono::seconds(10);
constexpr size_t kAlign       = 256;

using Clock = std::chrono::steady_clock;

// Free chunks for any thread; one not asked for within kPoolAge goes back to the device, the oldest ones when
// the bound is passed, all when an allocation fails. What keeps the time is a thread that lives as long as there
// are free chunks: a program that has ended its work leaves nothing on a device that others use.
class ChunkPool {
 public:
  ChunkPool() : pid(getpid()) {
    std::atexit([] { instance().stop_timer(); });  // (registered after the runtime's own, so it runs before)
  }
  static ChunkPool& instance() {
    static ChunkPool* p = new ChunkPool;  // never destroyed: systems may go after static destructors have run
    return *p;
  }
  // a chunk of at least want bytes on the device (its size in size), or none
  void* take(size_t want, int dev, size_t& size) {
    std::vector<void*> old;
    void* p = nullptr;
    {
      std::lock_guard<std::mutex> lock(m);
      expire(old);
      int best = -1;
      for (int i = 0; i < (int)free.size(); ++i)
        if (free[i].dev == dev && free[i].size >= want && free[i].size <= 8 * want &&
            (best < 0 || free[i].size < free[best].size))
          best = i;
      if (best >= 0) {
        p    = free[best].p;
        size = free[best].size;
        held -= size;
        free.erase(free.begin() + best);
      }
    }
    drop(old);
    return p;
  }
  void give(void* p, size_t size, int dev) {
    std::vector<void*> old;
    {
      std::lock_guard<std::mutex> lock(m);
      expire(old);
      free.push_back({p, size, dev, Clock::now()});
      held += size;
      while (held > kPoolBytes) pop_front(old);
      start_timer();
    }
    drop(old);
  }
  void clear() {
    std::vector<void*> old;
    {
      std::lock_guard<std::mutex> lock(m);
      while (!free.empty()) pop_front(old);
    }
    drop(old);
  }

 private:
  struct Entry {
    void* p;
    size_t size;
    int dev;
    Clock::time_point since;
  };
  void pop_front(std::vector<void*>& old) {
    old.push_back(free.front().p);
    held -= free.front().size;
    free.erase(free.begin());
  }
  void expire(std::vector<void*>& old) {
    const auto now = Clock::now();
    while (!free.empty() && now - free.front().since > kPoolAge) pop_front(old);
  }
  static void drop(const std::vector<void*>& old) {
    for (void* p : old) (void)hipFree(p);
  }
  // (m held) A thread that has ended has let go of m for good; a forked child has no such thread, and no device.
  void start_timer() {
    if (timed || stopped || free.empty() || getpid() != pid) return;
    if (timer.joinable()) timer.join();
    try {
      timer = std::thread([this] { run_timer(); });
      timed = true;
    } catch (const std::system_error&) {  // no thread to be had: chunks age with the next calls
    }
  }
  void run_timer() {
    // hipFree here must not end a capture that another thread has begun
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    std::unique_lock<std::mutex> lock(m);
    while (!stopped && !free.empty()) {
      wake.wait_until(lock, free.front().since + kPoolAge + std::chrono::milliseconds(1));
      std::vector<void*> old;
      if (!stopped) expire(old);
      lock.unlock();
      drop(old);
      lock.lock();
    }
    timed = false;
  }
  void stop_timer() {
    if (getpid() != pid) return;
    {
      std::lock_guard<std::mutex> lock(m);
      stopped = true;
    }
    wake.notify_all();
    if (timer.joinable()) timer.join();
  }
  std::mutex m;
  std::condition_variable wake;
  std::thread timer;
  const pid_t pid;
  bool timed = false, stopped = false;
  std::vector<Entry> free;  // oldest first
  size_t held = 0;
};

static ChunkPool& pool() { return ChunkPool::instance(); }

// null where the device has no room
static void* try_malloc(size_t bytes) {
  if (bytes > g_most) return nullptr;
  void* p      = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    pool().clear();
    e = hipMalloc(&p, bytes);
  }
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return nullptr;
  }
  CPPE_HIP_CHECK(e);
  return p;
}

void* device_malloc(size_t bytes) {
  void* p = try_malloc(bytes);
  if (!p) throw out_of_memory("out of device memory: " + std::to_string(bytes) + " bytes");
  return p;
}

// ---- arenas ----------------------------------------------------------------------------------
static thread_local DeviceArena* t_arena = nullptr;
DeviceArena* current_arena() { return t_arena; }

static size_t rounded(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

void* DeviceArena::take(size_t bytes) {
  const size_t need = rounded(bytes);
  if (bytes > g_most) throw out_of_memory("out of device memory: " + std::to_string(bytes) + " bytes");
  // the smallest hole that fits
  Chunk* at = nullptr;
  std::map<size_t, size_t>::iterator hole;
  for (Chunk& c : chunks)
    for (auto h = c.holes.begin(); h != c.holes.end(); ++h)
      if (h->second >= need && (!at || h->second < hole->second)) {
        at   = &c;
        hole = h;
      }
  if (!at) {
    size_t size = need;
    void* p     = nullptr;
    int dev     = 0;
    CPPE_HIP_CHECK(hipGetDevice(&dev));
    if (need <= kChunkPooled) {
      size = kChunkMin;
      while (size < need || (size < total && size < kChunkPooled)) size *= 2;
      if (size > g_most) size = need;
      p = pool().take(size, dev, size);
    }
    chunks.reserve(chunks.size() + 1);
    if (!p && size > need) p = try_malloc(size);
    if (!p) p = device_malloc(size = need);  // (no room to grow: what is asked for alone)
    chunks.push_back({static_cast<char*>(p), size, 0, dev, {}});
    total += size;
    at = &chunks.back();
    hole = at->holes.emplace(0, size).first;
  }
  const size_t off = hole->first, len = hole->second;
  at->holes.erase(hole);
  if (len > need) at->holes.emplace(off + need, len - need);
  at->used += need;
  return at->base + off;
}

void DeviceArena::give(void* p, size_t bytes) {
  const size_t len = rounded(bytes);
  for (size_t i = 0; i < chunks.size(); ++i) {
    Chunk& c = chunks[i];
    if (p < c.base || p >= c.base + c.size) continue;
    c.used -= len;
    if (c.used == 0 && c.size > kChunkPooled) {
      (void)hipFree(c.base);  // waits for the device
      total -= c.size;
      chunks.erase(chunks.begin() + i);
      return;
    }
    size_t off = static_cast<char*>(p) - c.base, end = off + len;
    auto next = c.holes.lower_bound(off);
    if (next != c.holes.end() && next->first == end) {
      end += next->second;
      next = c.holes.erase(next);
    }
    if (next != c.holes.begin()) {
      auto prev = std::prev(next);
      if (prev->first + prev->second == off) {
        prev->second = end - prev->first;
        return;
      }
    }
    c.holes.emplace(off, end - off);
    return;
  }
}

void DeviceArena::settle() {
  if (settled || chunks.empty()) return;
  settled = true;
  failed  = hipStreamSynchronize(stream) != hipSuccess;
}

DeviceArena::~DeviceArena() {
  settle();
  for (Chunk& c : chunks) {
    if (failed || c.size > kChunkPooled)
      (void)hipFree(c.base);
    else
      pool().give(c.base, c.size, c.dev);
  }
}

// ---- staging ---------------------------------------------------------------------------------
// One transfer uses half of a block's kSlots pinned slots (one half for each direction: filling a slot that
// the device wrote last runs at a tenth of the rate), filled and drained in turn while the copy engine works
// on the others. A block serves the transfers of one entry point (ArenaScope) and goes back to a list once
// its copies are done, which an entry point's results have waited for anyway; at most kBlocks are made in
// the process, and transfers beyond take the runtime's way. (No slot is left in use behind a call: an
// event whose stream is gone may not be asked.)
// Arrays below kStageMin gain nothing. From kStageMax on the runtime's pinning of the pages is faster than one
// thread that fills slots from memory beyond the caches (loss and gradient of 63,001 samples 1.2 ms, 1.8 through
// slots); 1 MiB takes 0.39 ms to the device the runtime's way and 0.09 through slots.
constexpr int kSlots       = 16, kHalf = kSlots / 2;
constexpr size_t kSlot     = size_t(256) << 10;
constexpr size_t kStageMin = size_t(48) << 10;
constexpr size_t kStageMax = size_t(3) << 20;
constexpr int kBlocks      = 4;

struct Staging {
  char* host = nullptr;
  int dev    = 0;
  hipEvent_t ev[kSlots] = {};
  bool busy[kSlots]     = {};
  int next[2]           = {};
  ~Staging() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (host) (void)hipHostFree(host);
  }
  // the next slot of a direction (0: to the device), no longer in use
  int slot(int dir) {
    const int s = dir * kHalf + next[dir];
    next[dir]   = (next[dir] + 1) % kHalf;
    wait(s);
    return s;
  }
  void wait(int s) {
    if (busy[s]) CPPE_HIP_CHECK(hipEventSynchronize(ev[s]));
    busy[s] = false;
  }
  void mark(int s, hipStream_t st) {
    CPPE_HIP_CHECK(hipEventRecord(ev[s], st));
    busy[s] = true;
  }
};

struct StagingList {
  std::mutex m;
  std::vector<std::unique_ptr<Staging>> free;
  int made = 0;
};
static StagingList& staging() {
  static StagingList* l = new StagingList;
  return *l;
}

// A block for this thread's device, taken with the first transfer; its destructor waits for the copies and
// gives it back (after an error the block is given up: its copies may still run).
class StagingUse {
 public:
  Staging* get() {
    if (b || tried) return b.get();
    tried   = true;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    StagingList& l = staging();
    {
      std::lock_guard<std::mutex> lock(l.m);
      for (size_t i = 0; i < l.free.size(); ++i)
        if (l.free[i]->dev == dev) {
          b = std::move(l.free[i]);
          l.free.erase(l.free.begin() + i);
          return b.get();
        }
      if (l.made == kBlocks) return nullptr;
      ++l.made;
    }
    auto n  = std::make_unique<Staging>();
    n->dev  = dev;
    bool ok = hipHostMalloc((void**)&n->host, kSlots * kSlot, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t& e : n->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) {
      b = std::move(n);
      return b.get();
    }
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(l.m);
    --l.made;
    return nullptr;
  }
  ~StagingUse() {
    if (!b) return;
    bool ok = true;
    for (int s = 0; s < kSlots; ++s) {
      if (b->busy[s]) ok = hipEventSynchronize(b->ev[s]) == hipSuccess && ok;
      b->busy[s] = false;
    }
    if (!ok) {
      (void)b.release();
      return;
    }
    std::lock_guard<std::mutex> lock(staging().m);
    staging().free.push_back(std::move(b));
  }

 private:
  std::unique_ptr<Staging> b;
  bool tried = false;
};

static thread_local StagingUse* t_slots = nullptr;

ArenaScope::ArenaScope(DeviceArena& a) : prev(t_arena) {
  if (!t_slots) {
    slots   = std::make_unique<StagingUse>();
    t_slots = slots.get();
  }
  t_arena = &a;
}
ArenaScope::~ArenaScope() {
  t_arena = prev;
  if (slots) t_slots = nullptr;
}

static bool stage_size(size_t bytes) { return bytes >= kStageMin && bytes < kStageMax; }

// Pinned memory needs no staging.
static bool pinned(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

void to_device(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return;
  if (stage_size(bytes) && !pinned(src)) {
    StagingUse own;
    if (Staging* b = (t_slots ? t_slots : &own)->get()) {
      for (size_t o = 0; o < bytes; o += kSlot) {
        const size_t len = std::min(kSlot, bytes - o);
        const int s      = b->slot(0);
        char* h          = b->host + s * kSlot;
        std::memcpy(h, static_cast<const char*>(src) + o, len);
        CPPE_HIP_CHECK(hipMemcpyAsync(static_cast<char*>(dst) + o, h, len, hipMemcpyHostToDevice, st));
        b->mark(s, st);
      }
      return;
    }
  }
  CPPE_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
}

void to_host(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes && stage_size(bytes) && !pinned(dst)) {
    StagingUse own;
    if (Staging* b = (t_slots ? t_slots : &own)->get()) {
      int at[kHalf];  // slots of the pieces in flight, oldest first from piece `out` on
      const size_t np = (bytes + kSlot - 1) / kSlot;
      size_t in = 0, out = 0;
      while (out < np) {
        for (; in < np && in - out < (size_t)kHalf; ++in) {
          const int s = b->slot(1);
          at[in % kHalf] = s;
          CPPE_HIP_CHECK(hipMemcpyAsync(b->host + s * kSlot, static_cast<const char*>(src) + in * kSlot,
                                        std::min(kSlot, bytes - in * kSlot), hipMemcpyDeviceToHost, st));
          b->mark(s, st);
        }
        const int s = at[out % kHalf];
        b->wait(s);
        std::memcpy(static_cast<char*>(dst) + out * kSlot, b->host + s * kSlot, std::min(kSlot, bytes - out * kSlot));
        ++out;
      }
      return;
    }
  }
  if (bytes) CPPE_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
  CPPE_HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace cppe_dev
