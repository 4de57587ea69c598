// A workgroup on the CPU, for tests of device headers: every lane is a fiber of
// one thread, a wavefront's lanes meet at its cross-lane operations and the
// workgroup's at __syncthreads().  Lanes run ahead as far as they can, one
// after another in the order of their wavefronts (reversed on request): an order
// that the hardware may take between wavefronts, and stricter than it within one.
// A workgroup whose lanes wait at different barriers ends with "barrier
// mismatch".
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#define __host__
#define __device__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)

struct double2 { double x, y; };
struct float2 { float x, y; };
struct float4 { float x, y, z, w; };
inline double2 make_double2(double x, double y) { return {x, y}; }
inline float2 make_float2(float x, float y) { return {x, y}; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }

namespace emu {

struct Lane {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack;
  int site = 0;      // where it waits: 0 runs, > 0 barrier (its line), < 0 cross-lane operation
  bool done = false;
  uint64_t slot = 0;  // operand of the cross-lane operation
};
struct Block {
  std::vector<Lane> lanes;
  std::function<void()> body;
  ucontext_t home;
  int cur = 0, dim = 0;
  std::string error;
};
inline Block* block = nullptr;
constexpr size_t kStack = 128 << 10;

inline void wait_at(int site) {
  Lane& l = block->lanes[block->cur];
  l.site = site;
  swapcontext(&l.ctx, &block->home);
}
inline void entry() {
  Lane& l = block->lanes[block->cur];
  block->body();
  l.done = true;
  swapcontext(&l.ctx, &block->home);
}

// Runs `body` on `threads` lanes; "" or what went wrong.
inline std::string run(int threads, bool reversed, std::function<void()> body) {
  Block b;
  b.dim = threads;
  b.body = std::move(body);
  b.lanes.resize(threads);
  block = &b;
  for (Lane& l : b.lanes) {
    l.stack.reset(new char[kStack]);
    getcontext(&l.ctx);
    l.ctx.uc_stack.ss_sp = l.stack.get();
    l.ctx.uc_stack.ss_size = kStack;
    l.ctx.uc_link = nullptr;
    makecontext(&l.ctx, entry, 0);
  }
  const int waves = threads / 64;
  for (bool left = true; left && b.error.empty();) {
    left = false;
    for (int k = 0; k < waves; ++k) {
      const int w = reversed ? waves - 1 - k : k;
      Lane* l = &b.lanes[64 * w];
      // this wavefront until it waits at a barrier or has ended
      for (;;) {
        for (int i = 0; i < 64; ++i)
          if (!l[i].done && !l[i].site) {
            b.cur = 64 * w + i;
            swapcontext(&b.home, &l[i].ctx);
          }
        // the lanes at a cross-lane operation (the others are past the branch
        // it stands in, at a barrier)
        int site = 0;
        for (int i = 0; i < 64; ++i)
          if (l[i].site < 0) {
            if (site && l[i].site != site) b.error = "lanes at different operations";
            site = l[i].site;
          }
        if (!site || !b.error.empty()) break;
        for (int i = 0; i < 64; ++i)
          if (l[i].site < 0) l[i].site = 0;
      }
    }
    int site = 0;
    for (Lane& l : b.lanes) {
      if (l.done) continue;
      left = true;
      if (site && l.site != site) b.error = "barrier mismatch";
      site = l.site;
    }
    for (Lane& l : b.lanes)
      if (left && l.done) b.error = "barrier mismatch";
    for (Lane& l : b.lanes) l.site = 0;
  }
  block = nullptr;
  return b.error;
}

// the operands of a wavefront's lanes, after all have given theirs; a second
// meeting keeps them until all have read
template <class T, class F>
inline T exchange(T v, int site, F&& pick) {
  static_assert(sizeof(T) <= 8, "one slot");
  const int me = block->cur, base = me & ~63;
  memcpy(&block->lanes[me].slot, &v, sizeof(T));
  wait_at(-2 * site);
  auto at = [&](int lane) {
    T r;
    memcpy(&r, &block->lanes[base + lane].slot, sizeof(T));
    return r;
  };
  const auto r = pick(at, me & 63);
  wait_at(-2 * site - 1);
  return r;
}

struct Idx {
  struct X {
    operator int() const { return block->cur; }
  } x;
};
struct BDim {
  struct X {
    operator int() const { return block->dim; }
  } x;
};

inline long reciprocal_roots = 0;  // calls of rsqrt

}  // namespace emu

inline emu::Idx threadIdx;
inline emu::BDim blockDim;
struct { int x = 0, y = 0, z = 0; } inline blockIdx;

#define __syncthreads() emu::wait_at(__LINE__)
inline void __threadfence_block() {}
template <class T>
inline T __shfl_xor(T v, int mask, int) {
  return emu::exchange(v, 1, [&](auto at, int lane) { return at(lane ^ mask); });
}
inline unsigned long long __ballot(bool p) {
  const int base = emu::block->cur & ~63;
  emu::block->lanes[emu::block->cur].slot = p;
  emu::wait_at(-4);
  unsigned long long m = 0;
  for (int i = 0; i < 64; ++i) m |= (unsigned long long)(emu::block->lanes[base + i].slot & 1) << i;
  emu::wait_at(-5);
  return m;
}
inline int __builtin_amdgcn_update_dpp(int, int v, int ctrl, int, int, bool) {
  return emu::exchange(v, 3, [&](auto at, int lane) {
    switch (ctrl) {
      case 0xB1: return at(lane ^ 1);
      case 0x4E: return at(lane ^ 2);
      case 0x141: return at(lane ^ 7);
      case 0x140: return at(lane ^ 15);
    }
    emu::block->error = "unknown DPP control";
    return 0;
  });
}
inline int __builtin_amdgcn_readlane(int v, int from) {
  return emu::exchange(v, 4, [&](auto at, int) { return at(from); });
}
inline int __builtin_amdgcn_readfirstlane(int v) { return __builtin_amdgcn_readlane(v, 0); }
inline long long __double_as_longlong(double v) {
  long long r;
  memcpy(&r, &v, 8);
  return r;
}
inline double __longlong_as_double(long long v) {
  double r;
  memcpy(&r, &v, 8);
  return r;
}
inline int __float_as_int(float v) {
  int r;
  memcpy(&r, &v, 4);
  return r;
}
inline float __int_as_float(int v) {
  float r;
  memcpy(&r, &v, 4);
  return r;
}
inline float __uint_as_float(unsigned v) { return __int_as_float((int)v); }
inline double __hiloint2double(int hi, int lo) {
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
inline int __ffsll(unsigned long long v) { return __builtin_ffsll((long long)v); }
inline int atomicMin(int* p, int v) {
  const int o = *p;
  *p = std::min(o, v);
  return o;
}
inline double rsqrt(double x) {
  ++emu::reciprocal_roots;
  return 1.0 / sqrt(x);
}
inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }

// named by the headers, not used here
struct emu_rsrc {};
#define __amdgpu_buffer_rsrc_t emu_rsrc
typedef unsigned emu_u2 __attribute__((ext_vector_type(2)));
typedef unsigned emu_u4 __attribute__((ext_vector_type(4)));
typedef double emu_d4 __attribute__((ext_vector_type(4)));
inline emu_rsrc __builtin_amdgcn_make_buffer_rsrc(void*, short, int, int) { return {}; }
inline emu_u2 __builtin_amdgcn_raw_buffer_load_b64(emu_rsrc, int, int, int) { return 0; }
inline emu_u4 __builtin_amdgcn_raw_buffer_load_b128(emu_rsrc, int, int, int) { return 0; }
inline emu_d4 __builtin_amdgcn_mfma_f64_16x16x4f64(double, double, emu_d4 c, int, int, int) {
  return c;
}
