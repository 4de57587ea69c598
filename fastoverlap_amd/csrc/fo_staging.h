// Pinned staging of small host transfers.
//
// A buffer is one caller's from get to put; at most kSlabsKept idle ones are
// kept.  One copy of a batch's adjacent outputs through a buffer takes 10 us; a
// copy of each output into pageable memory took 8..15 us apiece.  Larger transfers
// go to the caller's memory directly (18 GB/s, as fast as the copy out of a
// buffer).
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <vector>

namespace fo {

constexpr size_t kSlabBytes = 256 << 10;
constexpr size_t kSlabsKept = 16;

class SlabPool {
 public:
  void* get() {  // nullptr: the caller copies directly
    {
      std::lock_guard<std::mutex> g(mu_);
      if (!idle_.empty()) {
        void* p = idle_.back();
        idle_.pop_back();
        return p;
      }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, kSlabBytes, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    return p;
  }
  void put(void* p) {
    if (!p) return;
    {
      std::lock_guard<std::mutex> g(mu_);
      if (idle_.size() < kSlabsKept) {
        idle_.push_back(p);
        return;
      }
    }
    (void)hipHostFree(p);
  }
  void clear() {
    for (void* p : idle_) (void)hipHostFree(p);
    idle_.clear();
  }

 private:
  std::mutex mu_;
  std::vector<void*> idle_;
};

// The buffer that a batch's last host positions may still be copied from.  Calls
// on one batch may come from several threads (one sets the next positions while
// another reads the last results), so the buffer changes hands by exchange: it is
// stored after its copy has been queued, and who wants to give it back takes
// it out before waiting for the stream.  What was taken before a wait was queued
// before it and has been read when the wait ends; what another thread stores
// meanwhile stays.
using SlabSlot = std::atomic<void*>;

// Waits for the stream and gives the slot's buffer back.
inline hipError_t sync_staged(SlabPool& pool, SlabSlot& slot, hipStream_t s) {
  void* mine = slot.exchange(nullptr);
  const hipError_t e = hipStreamSynchronize(s);
  pool.put(mine);
  return e;
}

// Device memory read in one go: [dev, dev + bytes) through a staging buffer into
// `use(const char*)`, with the stream waited for and the slot's buffer given
// back.  False: nothing was done, the range has to be copied directly.
template <class F>
bool read_staged(SlabPool& pool, SlabSlot& slot, hipStream_t s, const void* dev, size_t bytes,
                 F&& use, hipError_t* err) {
  if (bytes > kSlabBytes) return false;
  void* slab = pool.get();
  if (!slab) return false;
  *err = hipMemcpyAsync(slab, dev, bytes, hipMemcpyDeviceToHost, s);
  const hipError_t e = sync_staged(pool, slot, s);
  if (*err == hipSuccess) *err = e;
  if (*err == hipSuccess) use((const char*)slab);
  pool.put(slab);
  return true;
}

// Two host arrays of `bytes` to dst and dst + gap as one copy, which is not
// waited for.  False: nothing was done, the arrays have to be copied directly.
inline bool write_staged(SlabPool& pool, SlabSlot& slot, hipStream_t s, void* dst, size_t gap,
                         const void* p1, const void* p2, size_t bytes, hipError_t* err) {
  if (gap + bytes > kSlabBytes) return false;
  void* slab = slot.exchange(nullptr);
  if (slab) {
    *err = hipStreamSynchronize(s);  // an earlier copy may still read it
  } else {
    slab = pool.get();
    if (!slab) return false;
    *err = hipSuccess;
  }
  if (*err == hipSuccess) {
    memcpy(slab, p1, bytes);
    memcpy((char*)slab + gap, p2, bytes);
    *err = hipMemcpyAsync(dst, slab, gap + bytes, hipMemcpyHostToDevice, s);
  }
  if (void* other = slot.exchange(slab)) {  // of another thread, in between
    const hipError_t e = hipStreamSynchronize(s);
    if (*err == hipSuccess) *err = e;
    pool.put(other);
  }
  return true;
}

}  // namespace fo
