// A workgroup of wave64 kernels on the CPU: every lane is a fiber, the lanes of a wave meet at each
// wave-wide operation and the waves at each barrier, and between those points a schedule decides which
// wave goes on. Device code compiled against this header (in place of hip/hip_runtime.h) runs as it is
// written, so a test can run one wave far ahead of the others between two barriers, which the GPU does
// only now and then.
//
// Reported as failures: lanes of a wave at different wave-wide operations, waves at different
// barriers, a lane that leaves while others wait for it, a permute from a lane above 63, a
// readfirstlane of values that differ. x86-64 only (the fiber switch).
//
// wave_slot (common.hpp) is the one wave-wide operation that kernels call with some of their lanes:
// programs define it as emu::slot, an add of the lane's own.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <initializer_list>
#include <memory>
#include <random>
#include <type_traits>
#include <vector>

namespace emu {

struct Index {
  unsigned x = 0, y = 0, z = 0;
};

extern "C" void emu_switch(void **save, void *to);
asm(R"(
.text
.globl emu_switch
.type emu_switch, @function
emu_switch:
  pushq %rbp
  pushq %rbx
  pushq %r12
  pushq %r13
  pushq %r14
  pushq %r15
  movq %rsp, (%rdi)
  movq %rsi, %rsp
  popq %r15
  popq %r14
  popq %r13
  popq %r12
  popq %rbx
  popq %rbp
  ret
.size emu_switch, .-emu_switch
)");

constexpr size_t kStack = 256 << 10;
enum State { kRunnable, kInWave, kAtBarrier, kDone };

struct Fiber {
  Index thread;
  int lane = 0, wave = 0;
  State state = kRunnable;
  const char *file = "";
  int line = 0;     // where it waits
  unsigned ops = 0;  // wave-wide operations so far
  void *sp = nullptr;
  std::unique_ptr<char[]> stack;
};
struct Wave {
  unsigned long long value[2][64];
  int waiting = 0;
};

struct Group {
  std::vector<Fiber> fibers;
  std::vector<Wave> waves;
  int at_barrier = 0, live = 0, value = 0, voted = 0;
  Fiber *now = nullptr;
  void *home = nullptr;
  const std::function<void()> *kernel = nullptr;
};
inline Group *group = nullptr;
inline Fiber &here() { return *group->now; }

[[noreturn]] inline void fail(const char *what, const Fiber &a, const Fiber &b) {
  std::printf("%s: thread %u at %s:%d, thread %u at %s:%d\n", what, a.thread.x, a.file, a.line, b.thread.x, b.file, b.line);
  std::fflush(stdout);
  std::_Exit(1);
}

inline void leave(Fiber &f) { emu_switch(&f.sp, group->home); }

// All 64 lanes of the caller's wave meet here.
inline void meet(const char *file, int line) {
  Fiber &f = here();
  Wave &w = group->waves[size_t(f.wave)];
  f.file = file;
  f.line = line;
  f.state = kInWave;
  if (++w.waiting == 64) {
    Fiber *first = &group->fibers[size_t(f.wave) * 64];
    for (int l = 0; l < 64; ++l) {
      if (first[l].state != kInWave || first[l].line != line || std::strcmp(first[l].file, file)) fail("a wave's lanes apart", first[l], f);
      first[l].state = kRunnable;
    }
    w.waiting = 0;
  }
  leave(f);
}

// The lanes' values of one operation, until the wave's next but one.
inline const unsigned long long *exchange(unsigned long long v, const char *file, int line) {
  Fiber &f = here();
  unsigned long long *slots = group->waves[size_t(f.wave)].value[f.ops++ & 1];
  slots[f.lane] = v;
  meet(file, line);
  return slots;
}

inline int barrier(int vote, const char *file, int line) {
  Fiber &f = here();
  f.file = file;
  f.line = line;
  f.state = kAtBarrier;
  group->voted |= vote;
  if (++group->at_barrier == int(group->fibers.size())) {
    for (Fiber &o : group->fibers) {
      if (o.line != line || std::strcmp(o.file, file)) fail("waves at different barriers", o, f);
      o.state = kRunnable;
    }
    group->at_barrier = 0;
    group->value = group->voted;
    group->voted = 0;
  }
  leave(f);
  return group->value;
}

inline void entry() {
  (*group->kernel)();
  Fiber &f = here();
  f.state = kDone;
  --group->live;
  for (;;) leave(f);
}

// Which wave goes on: the first runnable one of `order`, or (order empty) a random one at each
// meeting of lanes.
struct Schedule {
  std::vector<int> order;
  unsigned seed = 0;
};

// Runs one workgroup of `threads` (whole waves).
inline void run(int threads, const Schedule &schedule, const std::function<void()> &kernel) {
  Group g;
  g.fibers.resize(size_t(threads));
  g.waves.resize(size_t(threads) / 64);
  g.live = threads;
  g.kernel = &kernel;
  group = &g;
  for (int t = 0; t < threads; ++t) {
    Fiber &f = g.fibers[size_t(t)];
    f.thread.x = unsigned(t);
    f.lane = t & 63;
    f.wave = t >> 6;
    f.stack.reset(new char[kStack]);
    uintptr_t top = (uintptr_t(f.stack.get()) + kStack) & ~uintptr_t(15);
    void **sp = reinterpret_cast<void **>(top) - 2;  // entry's return address slot: aligned as after a call
    *sp = reinterpret_cast<void *>(&entry);
    f.sp = sp - 6;
    std::memset(f.sp, 0, 6 * sizeof(void *));
  }
  std::mt19937 rng(schedule.seed);
  const int waves = threads / 64;
  std::vector<int> order(schedule.order);
  auto runnable = [&](int w) {
    for (int l = 0; l < 64; ++l)
      if (g.fibers[size_t(w) * 64 + size_t(l)].state == kRunnable) return true;
    return false;
  };
  while (g.live) {
    int w = -1;
    if (order.empty()) {
      const int from = int(rng() % unsigned(waves));
      for (int i = 0; i < waves && w < 0; ++i)
        if (runnable((from + i) % waves)) w = (from + i) % waves;
    } else {
      for (int i : order)
        if (runnable(i)) { w = i; break; }
    }
    if (w < 0) {
      const Fiber *a = nullptr, *b = nullptr;
      for (const Fiber &f : g.fibers) {
        if (f.state == kAtBarrier) a = &f;
        if (f.state == kInWave || f.state == kDone) b = &f;
      }
      fail("no lane can go on", a ? *a : g.fibers[0], b ? *b : g.fibers[0]);
    }
    for (int l = 0; l < 64; ++l) {
      Fiber &f = g.fibers[size_t(w) * 64 + size_t(l)];
      if (f.state != kRunnable) continue;
      g.now = &f;
      emu_switch(&g.home, f.sp);
    }
  }
  group = nullptr;
}

inline unsigned long long ballot(bool b, const char *file, int line) {
  const unsigned long long *v = exchange(b, file, line);
  unsigned long long m = 0;
  for (int l = 0; l < 64; ++l) m |= (v[l] & 1ULL) << l;
  return m;
}
template <class T> T from_bits(unsigned long long b) {
  T v;
  std::memcpy(&v, &b, sizeof(T));
  return v;
}
template <class T> unsigned long long to_bits(T v) {
  unsigned long long b = 0;
  std::memcpy(&b, &v, sizeof(T));
  return b;
}
template <class T> T from_lane(T v, int lane, const char *file, int line) {
  const unsigned long long *s = exchange(to_bits(v), file, line);
  if (lane < 0 || lane > 63) fail("a value from a lane above 63", here(), here());
  return from_bits<T>(s[lane]);
}
inline int permute(int byte, int v, const char *file, int line) { return from_lane(v, byte >> 2, file, line); }
inline int uniform(int v, const char *file, int line) {
  const unsigned long long *s = exchange(to_bits(v), file, line);
  for (int l = 0; l < 64; ++l)
    if (s[l] != s[0]) fail("a readfirstlane of values that differ", here(), here());
  return v;
}
inline int dpp(int v, int control, const char *file, int line) {
  const int lane = here().lane;
  int from = -1;
  if (control == 0xB1) from = lane ^ 1;
  if (control == 0x4E) from = lane ^ 2;
  if (control == 0x141) from = lane ^ 7;
  if (control == 0x140) from = lane ^ 15;
  return from_lane(v, from, file, line);
}
inline int swizzle(int v, int control, const char *file, int line) {
  return from_lane(v, control == 0x401F ? here().lane ^ 16 : -1, file, line);
}
template <class T> T neighbour(T v, int from, const char *file, int line) {  // a shuffle that keeps its own value past the ends
  return from_lane(v, from < 0 || from > 63 ? here().lane : from, file, line);
}
inline int below(unsigned m, int base, int high) {
  const unsigned long long mask = (1ULL << here().lane) - 1ULL;
  return base + __builtin_popcount(m & unsigned(high ? mask >> 32 : mask));
}
inline int slot(int *counter) { return (*counter)++; }

template <class T, class F> T update(T *p, F &&f) {
  const T old = *p;
  *p = f(old);
  return old;
}

}  // namespace emu

#define __device__
#define __host__
#define __global__
#define __constant__
#define __shared__ thread_local
#define __forceinline__ inline
#define __launch_bounds__(...)
#define threadIdx (::emu::here().thread)
#define blockDim (::emu::Index{unsigned(::emu::group->fibers.size()), 1, 1})
#define blockIdx (::emu::Index{})

#define __syncthreads() ::emu::barrier(0, __FILE__, __LINE__)
#define __syncthreads_or(v) ::emu::barrier(v, __FILE__, __LINE__)
#define __ballot(b) ::emu::ballot(b, __FILE__, __LINE__)
#define __shfl(v, lane, width) ::emu::from_lane(v, lane, __FILE__, __LINE__)
#define __shfl_xor(v, mask, width) ::emu::from_lane(v, ::emu::here().lane ^ (mask), __FILE__, __LINE__)
#define __shfl_up(v, by, width) ::emu::neighbour(v, ::emu::here().lane - int(by), __FILE__, __LINE__)
#define __shfl_down(v, by, width) ::emu::neighbour(v, ::emu::here().lane + int(by), __FILE__, __LINE__)
#define __lane_id() (::emu::here().lane)
#define __builtin_amdgcn_ballot_w64(b) ::emu::ballot(b, __FILE__, __LINE__)
#define __builtin_amdgcn_ds_bpermute(byte, v) ::emu::permute(byte, v, __FILE__, __LINE__)
#define __builtin_amdgcn_ds_swizzle(v, control) ::emu::swizzle(v, control, __FILE__, __LINE__)
#define __builtin_amdgcn_update_dpp(old, v, control, rows, banks, bound) ::emu::dpp(v, control, __FILE__, __LINE__)
#define __builtin_amdgcn_readlane(v, lane) ::emu::from_lane(v, lane, __FILE__, __LINE__)
#define __builtin_amdgcn_readfirstlane(v) ::emu::uniform(v, __FILE__, __LINE__)
#define __builtin_amdgcn_mbcnt_lo(m, base) ::emu::below(m, base, 0)
#define __builtin_amdgcn_mbcnt_hi(m, base) ::emu::below(m, base, 1)
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() ::emu::meet(__FILE__, __LINE__)
#define wall_clock64() 0LL

#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __HIP_MEMORY_SCOPE_AGENT 1
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, v, order, scope) ((void)(*(p) = (v)))
#define __hip_atomic_fetch_add(p, v, order, scope) ::emu::update(p, [&](auto o) { return o + (v); })
#define __hip_atomic_fetch_sub(p, v, order, scope) ::emu::update(p, [&](auto o) { return o - (v); })
#define __hip_atomic_fetch_min(p, v, order, scope) ::emu::update(p, [&](auto o) { return o < (v) ? o : (v); })
#define __hip_atomic_fetch_max(p, v, order, scope) ::emu::update(p, [&](auto o) { return o > (v) ? o : (v); })
#define __hip_atomic_fetch_and(p, v, order, scope) ::emu::update(p, [&](auto o) { return o & (v); })
#define __hip_atomic_fetch_or(p, v, order, scope) ::emu::update(p, [&](auto o) { return o | (v); })
#define __hip_atomic_exchange(p, v, order, scope) ::emu::update(p, [&](auto) { return v; })
#define __hip_atomic_compare_exchange_strong(p, expected, desired, success, failure, scope) \
  (void)(*(p) == *(expected) ? (*(p) = (desired), true) : (*(expected) = *(p), false))

template <class T> T atomicAdd(T *p, T v) { return ::emu::update(p, [&](T o) { return T(o + v); }); }
template <class T> T atomicOr(T *p, T v) { return ::emu::update(p, [&](T o) { return T(o | v); }); }
template <class T> T atomicMin(T *p, T v) { return ::emu::update(p, [&](T o) { return o < v ? o : v; }); }
template <class T> T atomicMax(T *p, T v) { return ::emu::update(p, [&](T o) { return o > v ? o : v; }); }
template <class T> T atomicCAS(T *p, T expected, T v) { return ::emu::update(p, [&](T o) { return o == expected ? v : o; }); }

inline int __float_as_int(float f) { return emu::from_bits<int>(emu::to_bits(f)); }
inline unsigned __float_as_uint(float f) { return emu::from_bits<unsigned>(emu::to_bits(f)); }
inline float __int_as_float(int v) { return emu::from_bits<float>(emu::to_bits(v)); }
inline float __uint_as_float(unsigned v) { return emu::from_bits<float>(emu::to_bits(v)); }
inline int __popc(unsigned v) { return __builtin_popcount(v); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __ffs(int v) { return __builtin_ffs(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
inline int __clz(int v) { return v ? __builtin_clz(unsigned(v)) : 32; }
inline int __clzll(long long v) { return v ? __builtin_clzll((unsigned long long)v) : 64; }
using std::max;
using std::min;

struct int2 { int x, y; };
struct int3 { int x, y, z; };
struct int4 { int x, y, z, w; };
inline int2 make_int2(int x, int y) { return int2{x, y}; }
inline int4 make_int4(int x, int y, int z, int w) { return int4{x, y, z, w}; }

// What the host headers name.
enum hipError_t { hipSuccess = 0 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipMemcpyDefault };
using hipStream_t = void *;
using hipEvent_t = void *;
using std::isinf;
inline const char *hipGetErrorString(hipError_t) { return ""; }
template <class... A> hipError_t emu_host_call(A...) { return hipSuccess; }
#define hipSetDevice emu_host_call
#define hipGetDevice emu_host_call
#define hipGetLastError emu_host_call<>
#define hipStreamSynchronize emu_host_call
#define hipEventCreate emu_host_call
#define hipEventRecord emu_host_call
#define hipEventSynchronize emu_host_call
#define hipEventElapsedTime emu_host_call
#define hipEventDestroy emu_host_call
#define hipMemsetAsync emu_host_call
#define hipMemcpyAsync emu_host_call
