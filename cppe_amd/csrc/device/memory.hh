// Device memory of a system and transfers of pageable host memory.
//
// What bounds a short run is the host: hipMalloc and hipFree of blocks of a MiB and more take 30 to 330 us
// each (smaller ones 1 us, from the runtime's own pool, but 280 us where that pool has just been emptied by
// the last system's end and is mapped again), a system makes some 90, and the runtime copies
// pageable arrays of 64 KiB to 3 MiB at 2.9 GB/s. So blocks of kArenaMin and more come from chunks a system
// keeps (DeviceArena), chunks outlive it in a bounded pool, and such arrays go through pinned slots: the static
// fields and energies of 120,000 sites, system included, took 15.2 ms and now 5.4, a geometry step of 24,000
// sites 15.9 and 8.4, the loss and gradient of 63,001 samples (arena alone) 1.18 and 1.02.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <map>
#include <memory>
#include <utility>
#include <vector>

#include "common.hh"

namespace cppe_dev {

// hipMalloc that empties the chunk pool and tries again before it gives up (throws out_of_memory).
void* device_malloc(size_t bytes);

// Blocks of one owner whose work is all ordered on one stream (others join it): a block given back may be
// taken again at once, as what used it comes before in that order. Used by one thread at a time, as its owner.
class DeviceArena {
 public:
  // Smaller blocks come from the runtime's own pool. With 512 KiB here a geometry step of 24,000 sites mapped
  // that pool anew once or twice in each pass: 8.9 to 9.7 ms, 8.3 to 8.5 with 64 (and with 16).
  static constexpr size_t kArenaMin = size_t(1) << 16;
  explicit DeviceArena(hipStream_t st = nullptr) : stream(st) {}
  DeviceArena(const DeviceArena&) = delete;
  DeviceArena& operator=(const DeviceArena&) = delete;
  ~DeviceArena();
  void* take(size_t bytes);
  void give(void* p, size_t bytes);
  // Waits for the owner's stream, before its chunks can serve another one (the owner calls it before the
  // stream goes; else the destructor does).
  void settle();
  hipStream_t stream;

 private:
  struct Chunk {
    char* base;
    size_t size, used;
    int dev;
    std::map<size_t, size_t> holes;  // offset -> bytes
  };
  std::vector<Chunk> chunks;
  size_t total = 0;
  bool settled = false, failed = false;
};

// While it lives, the dbufs this thread allocates come from the arena (the inner scope counts), and its
// transfers share one block of pinned slots (the outer scope's). The streams of both outlive the scope.
class StagingUse;
class ArenaScope {
 public:
  explicit ArenaScope(DeviceArena& a);
  ~ArenaScope();
  ArenaScope(const ArenaScope&) = delete;
  ArenaScope& operator=(const ArenaScope&) = delete;

 private:
  DeviceArena* prev;
  std::unique_ptr<StagingUse> slots;
};
DeviceArena* current_arena();

// Device buffer with RAII release.
template <typename T>
struct dbuf {
  T* p = nullptr;
  size_t n = 0;
  dbuf() = default;
  dbuf(const dbuf&) = delete;
  dbuf& operator=(const dbuf&) = delete;
  ~dbuf() { release(); }
  void release() {
    if (arena)
      arena->give(p, n * sizeof(T));
    else if (p)
      (void)hipFree(p);
    p = nullptr;
    n = 0;
    arena = nullptr;
  }
  void alloc(size_t count) {
    if (count <= n && p) return;
    release();
    if (count == 0) count = 1;
    DeviceArena* a = count * sizeof(T) >= DeviceArena::kArenaMin ? current_arena() : nullptr;
    p     = static_cast<T*>(a ? a->take(count * sizeof(T)) : device_malloc(count * sizeof(T)));
    arena = a;
    n     = count;
  }
  void swap(dbuf& o) {
    std::swap(p, o.p);
    std::swap(n, o.n);
    std::swap(arena, o.arena);
  }
  void zero(hipStream_t s) { CPPE_HIP_CHECK(hipMemsetAsync(p, 0, n * sizeof(T), s)); }
  operator T*() const { return p; }

 private:
  DeviceArena* arena = nullptr;  // whose block this is (none: hipMalloc's)
};

// Copies on a stream from and to host memory of any kind. to_device returns once pageable src may change; pinned src
// must stay as it is until the stream has passed the copy (every entry point waits for its stream before it returns).
// to_host returns once dst holds the data.
void to_device(void* dst, const void* src, size_t bytes, hipStream_t st);
void to_host(void* dst, const void* src, size_t bytes, hipStream_t st);

}  // namespace cppe_dev
