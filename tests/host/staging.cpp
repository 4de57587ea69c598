// The staging buffers (fo_staging.h) with a runtime whose copies happen at the
// next wait, and calls of a second thread placed where they do most harm: right
// after another call's wait.  Prints "ok" or what went wrong.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>

#include <functional>
#include <set>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
constexpr int hipHostMallocDefault = 0;
struct Stream {
  std::vector<std::function<void()>> queue;
  std::function<void()> after_wait;  // once
};
using hipStream_t = Stream*;
static std::set<void*> pinned;
static hipError_t hipHostMalloc(void** p, size_t n, int) {
  *p = calloc(1, n);
  pinned.insert(*p);
  return hipSuccess;
}
static int bad_frees = 0;
static hipError_t hipHostFree(void* p) {
  if (!pinned.erase(p)) {
    ++bad_frees;
    return hipErrorUnknown;
  }
  free(p);
  return hipSuccess;
}
static hipError_t hipGetLastError() { return hipSuccess; }
static hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  q->queue.push_back([=] { memcpy(d, s, n); });
  return hipSuccess;
}
static hipError_t hipStreamSynchronize(hipStream_t q) {
  for (auto& f : q->queue) f();
  q->queue.clear();
  auto f = std::move(q->after_wait);
  q->after_wait = nullptr;
  if (f) f();
  return hipSuccess;
}

#include "fo_staging.h"

struct Batch {
  fo::SlabSlot slab{nullptr};
  Stream s;
  double pos[6] = {0, 0, 0, 0, 0, 0};  // pos1, pos2, outputs
  void write(fo::SlabPool& pool, double a, double b) {
    const double p1[2] = {a, a}, p2[2] = {b, b};
    hipError_t e;
    if (!fo::write_staged(pool, slab, &s, pos, sizeof(p1), p1, p2, sizeof(p1), &e) || e)
      printf("write failed\n"), exit(1);
  }
  double read(fo::SlabPool& pool) {
    double out = 0;
    hipError_t e;
    if (!fo::read_staged(pool, slab, &s, pos + 4, 2 * sizeof(double),
                         [&](const char* h) { memcpy(&out, h, sizeof(out)); }, &e) ||
        e)
      printf("read failed\n"), exit(1);
    return out;
  }
};

int main() {
  fo::SlabPool pool;
  {
    // the next positions are set while the last results are read
    Batch a, b, c;
    a.write(pool, 1, 2);
    a.s.after_wait = [&] { a.write(pool, 3, 4); };
    a.read(pool);
    b.write(pool, 5, 6);  // other batches, from the same pool
    c.write(pool, 7, 8);
    fo::sync_staged(pool, a.slab, &a.s);
    fo::sync_staged(pool, b.slab, &b.s);
    fo::sync_staged(pool, c.slab, &c.s);
    if (a.pos[0] != 3 || a.pos[2] != 4) return printf("positions %g %g of another batch\n", a.pos[0], a.pos[2]), 1;
    if (b.pos[0] != 5 || b.pos[2] != 6) return printf("second batch %g %g\n", b.pos[0], b.pos[2]), 1;
  }
  {
    // two threads read one batch: its buffer goes back once
    Batch a, b, c;
    a.write(pool, 1, 2);
    a.s.after_wait = [&] { a.read(pool); };
    a.read(pool);
    b.write(pool, 5, 6);
    c.write(pool, 7, 8);
    fo::sync_staged(pool, b.slab, &b.s);
    fo::sync_staged(pool, c.slab, &c.s);
    if (b.pos[0] != 5 || c.pos[0] != 7) return printf("one buffer for two batches\n"), 1;
  }
  {
    // two threads set the positions of one batch: both copies leave whole
    Batch a, b;
    a.write(pool, 1, 2);
    a.s.after_wait = [&] { a.write(pool, 3, 4); };
    a.write(pool, 5, 6);
    b.write(pool, 7, 8);
    fo::sync_staged(pool, a.slab, &a.s);
    fo::sync_staged(pool, b.slab, &b.s);
    if (a.pos[0] != 5 || a.pos[2] != 6 || b.pos[0] != 7) return printf("two writers\n"), 1;
  }
  // a pool of idle buffers: bounded, each freed once
  std::vector<void*> held;
  for (size_t i = 0; i < 2 * fo::kSlabsKept; ++i) held.push_back(pool.get());
  if (std::set<void*>(held.begin(), held.end()).size() != held.size()) return printf("a buffer twice\n"), 1;
  for (void* p : held) pool.put(p);
  if (pinned.size() != fo::kSlabsKept) return printf("%zu idle buffers\n", pinned.size()), 1;
  pool.clear();
  if (bad_frees || !pinned.empty()) return printf("frees\n"), 1;
  printf("ok\n");
}
