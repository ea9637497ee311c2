// Shared device helpers for the gfx950 kernels: neighbour tables, coherent loads, float tricks.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace brook {

// 26-neighbour offsets in the reference's fixed order (faces, xy/yz/xz edges, corners;
// common.cuh:33-47). Every flood, walk and invalidation visits neighbours in this order.
__constant__ static const int kNX[26] = {-1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, -1, -1, 1, 1, -1, -1, -1, -1, 1, 1, 1, 1};
__constant__ static const int kNY[26] = {0, 0, -1, 1, 0, 0, -1, 1, -1, 1, -1, -1, 1, 1, 0, 0, 0, 0, -1, -1, 1, 1, -1, -1, 1, 1};
__constant__ static const int kNZ[26] = {0, 0, 0, 0, -1, 1, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1};
// Rank of neighbour k in dijkstra3d's order and its inverse (common.cuh:74-81); opposite offsets.
__constant__ static const int kD3Rank[26] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 21, 20, 24, 19, 23, 22, 25};
__constant__ static const int kD3Inv[26] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 22, 20, 19, 24, 23, 21, 25};
__constant__ static const int kOpp[26] = {1, 0, 3, 2, 5, 4, 9, 8, 7, 6, 13, 12, 11, 10, 17, 16, 15, 14, 25, 24, 23, 22, 21, 20, 19, 18};

// The same table as compile-time constants, for fully unrolled neighbour loops.
constexpr int kDX[26] = {-1, 1, 0, 0, 0, 0, -1, -1, 1, 1, 0, 0, 0, 0, -1, -1, 1, 1, -1, -1, -1, -1, 1, 1, 1, 1};
constexpr int kDY[26] = {0, 0, -1, 1, 0, 0, -1, 1, -1, 1, -1, -1, 1, 1, 0, 0, 0, 0, -1, -1, 1, 1, -1, -1, 1, 1};
constexpr int kDZ[26] = {0, 0, 0, 0, -1, 1, 0, 0, 0, 0, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1, -1, 1};
// The same deltas packed two bits per neighbour (delta + 1), for loops whose k is a run-time value:
// shifts of an immediate instead of table loads.
constexpr unsigned long long pack_deltas(const int (&t)[26]) {
  unsigned long long p = 0;
  for (int k = 0; k < 26; ++k) p |= (unsigned long long)(t[k] + 1) << (2 * k);
  return p;
}
constexpr unsigned long long kPackDX = pack_deltas(kDX), kPackDY = pack_deltas(kDY), kPackDZ = pack_deltas(kDZ);
constexpr int unpack_delta(unsigned long long p, int k) { return int((p >> (2 * k)) & 3ULL) - 1; }
constexpr bool deltas_match() {
  for (int k = 0; k < 26; ++k)
    if (unpack_delta(kPackDX, k) != kDX[k] || unpack_delta(kPackDY, k) != kDY[k] || unpack_delta(kPackDZ, k) != kDZ[k])
      return false;
  return true;
}
static_assert(deltas_match(), "packed neighbour deltas");
__device__ __forceinline__ int nb_dx(int k) { return unpack_delta(kPackDX, k); }
__device__ __forceinline__ int nb_dy(int k) { return unpack_delta(kPackDY, k); }
__device__ __forceinline__ int nb_dz(int k) { return unpack_delta(kPackDZ, k); }

constexpr float kInf = __builtin_huge_valf();
constexpr unsigned long long kMaxKey = ~0ULL;

struct Dims {
  int sx, sy, sz;
};

__device__ __forceinline__ void unravel(int v, const Dims &d, int &x, int &y, int &z) {
  int sxy = d.sx * d.sy;
  z = v / sxy;
  int r = v - z * sxy;
  y = r / d.sx;
  x = r - y * d.sx;
}
__device__ __forceinline__ bool inside(int x, int y, int z, const Dims &d) {
  return (unsigned)x < (unsigned)d.sx && (unsigned)y < (unsigned)d.sy && (unsigned)z < (unsigned)d.sz;
}
__device__ __forceinline__ int flat(int x, int y, int z, const Dims &d) { return x + d.sx * (y + d.sy * z); }
// Flat offset of neighbour k (only meaningful where its mask bit says it is inside the volume).
template <int K> __device__ __forceinline__ int nb_offset(const Dims &d) {
  return kDX[K] + d.sx * (kDY[K] + d.sy * kDZ[K]);
}
__device__ __forceinline__ int nb_offset(int k, const Dims &d) { return kNX[k] + d.sx * (kNY[k] + d.sy * kNZ[k]); }

// Calls f(integral_constant k) for k = B..E-1 with k known at compile time.
template <int B, int E, class F> __device__ __forceinline__ void for_nb(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    for_nb<B + 1, E>(f);
  }
}
template <class F> __device__ __forceinline__ void for_each_nb(F &&f) { for_nb<0, 26>(f); }

// ---- device-memory access in the global address space -------------------------------------------
// Pointers that reach a kernel inside a struct are generic, and generic accesses compile to FLAT
// instructions, which also count against the LDS counter (so every LDS wait waits for them too)
// and cannot use a scalar base. The kernels access device memory through the forms below, which
// name the global address space: plain loads and stores, and relaxed agent-scope atomics (the
// semantics of HIP's atomicX functions).
template <class T> __device__ __forceinline__ __attribute__((address_space(1))) T *gp(T *p) {
  return (__attribute__((address_space(1))) T *)p;
}
template <class T> struct same_type { using type = T; };
template <class T> using same_t = typename same_type<T>::type;
template <class T> __device__ __forceinline__ T g_ld(const T *p) { return *gp(p); }
template <class T> __device__ __forceinline__ void g_st(T *p, same_t<T> v) { *gp(p) = v; }
template <class T> __device__ __forceinline__ T g_min(T *p, same_t<T> v) {
  return __hip_atomic_fetch_min(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ T g_add(T *p, same_t<T> v) {
  return __hip_atomic_fetch_add(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ T g_or(T *p, same_t<T> v) {
  return __hip_atomic_fetch_or(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ T g_and(T *p, same_t<T> v) {
  return __hip_atomic_fetch_and(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Compare-and-swap; returns the previous value.
template <class T> __device__ __forceinline__ T g_cas(T *p, same_t<T> expected, same_t<T> desired) {
  __hip_atomic_compare_exchange_strong(gp(p), &expected, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return expected;
}

// Loads of memory that other threads change inside the same kernel: relaxed, agent scope, so the
// access is served by L2 (the CU's vector L1 may hold a stale line otherwise).
__device__ __forceinline__ int ld_i(const int *p) { return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned ld_u(const unsigned *p) { return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned long long ld_u64(const unsigned long long *p) {
  return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned char ld_u8(const unsigned char *p) {
  return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_i(int *p, int v) { __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Loads and stores of per-voxel data that, during one kernel, only the workgroup owning the voxel's
// component label touches (floods, tracer): workgroup scope is all the memory model needs, and the
// accesses may then be served by the CU's vector L1 instead of always going to L2.
#ifndef BROOK_LABEL_SCOPE
#define BROOK_LABEL_SCOPE __HIP_MEMORY_SCOPE_WORKGROUP
#endif
__device__ __forceinline__ int lp_i(const int *p) { return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, BROOK_LABEL_SCOPE); }
__device__ __forceinline__ unsigned long long lp_u64(const unsigned long long *p) {
  return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, BROOK_LABEL_SCOPE);
}
__device__ __forceinline__ void sp_u64(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, BROOK_LABEL_SCOPE);
}

// Slot in a list whose length lives at *counter (any address space), for every lane that calls
// this at the same point: one atomic per wave, lanes numbered in lane order.
__device__ __forceinline__ int wave_slot(int *counter) {
  const unsigned long long act = __ballot(1);
  const int lane = __lane_id();
  const int leader = __ffsll((long long)act) - 1;
  int base = 0;
  if (lane == leader) base = atomicAdd(counter, __popcll(act));
  base = __shfl(base, leader, 64);
  return base + __popcll(act & ((1ULL << lane) - 1ULL));
}

// What the floods and the tracer touch per voxel, in three arrays, so that each phase's neighbour
// walk reads 8 bytes per neighbour:
//   mask   u32, bits [0, 26): the neighbours of the voxel's own nonzero id (0 for background)
//   road   u64, floods and railroad: distance (31 bits: a float's without its sign, which is 0) << 33
//          | far listed << 32 | not queued << 31 | cost (the PDRF's 31 bits; rails 0). One load gives a
//          neighbour's cost and its distance, and words of one voxel, whose cost is the same, order
//          by (distance, flags), so one atomic minimum both improves the distance and tells what
//          the voxel was. Unreached: distance +inf, not queued, so a candidate of infinite cost never
//          improves one.
//   claim  u64, invalidation: bottleneck << 32 | (source + 1) << 1 | queued; kDead (low half 0, which
//          no claim has) once the voxel is invalidated, kFree while it is alive and unclaimed.
// Background words of road and claim are never written, and both arrays have word_pad() words before
// and after the volume's, so a neighbour walk loads all 26 neighbours' words and lets the mask bits,
// which arrive beside them, say which count.
constexpr unsigned kCostBits = 0x7FFFFFFFu;
constexpr unsigned kInfBits = 0x7F800000u;
constexpr unsigned long long kNotQueued = 1ULL << 31, kFarListed = 1ULL << 32;
constexpr unsigned long long kUnreached = ((unsigned long long)kInfBits << 33) | kNotQueued;  // or'ed with the cost
__host__ __device__ constexpr unsigned road_dist(unsigned long long w) { return unsigned(w >> 33); }
__host__ __device__ constexpr unsigned road_cost(unsigned long long w) { return unsigned(w) & kCostBits; }
__host__ __device__ constexpr unsigned long long road_word(unsigned dist, unsigned long long flags, unsigned cost) {
  return ((unsigned long long)dist << 33) | flags | cost;
}
constexpr unsigned long long kFloodFree = kUnreached | kCostBits;  // the floods' words (no cost yet)

constexpr unsigned long long kDead = 0ULL, kFree = ~0ULL;

// The place of a step (dx, dy, dz) of up to one voxel from the word it starts at. Along a dimension of
// one voxel no mask bit leads anywhere and the step has no length, so that a flat volume needs no plane of
// padding on each side (two arrays of three times its words).
__host__ __device__ constexpr int step_offset(const Dims &d, int dx, int dy, int dz) {
  return dx + (d.sy > 1 ? d.sx * dy : 0) + (d.sz > 1 ? d.sx * d.sy * dz : 0);
}
constexpr long long word_pad(const Dims &d) {
  return (d.sz > 1 ? (long long)d.sx * d.sy : 0) + (d.sy > 1 ? d.sx : 0) + 1;  // the longest step
}
// Volumes whose padded words lie within 32-bit byte offsets: the kernels' narrow form, which adds a
// 32-bit offset per lane to a scalar base instead of computing 64-bit addresses.
constexpr bool narrow_words(const Dims &d) {
  return (long long)d.sx * d.sy * d.sz + 2 * word_pad(d) <= (1LL << 29);
}

// Division of 0 <= n < 2^31 by a constant d >= 1 as a high product and a shift: with 2^l the power
// of two at or above d and m = ceil(2^(31 + l) / d) < 2^32, m * d exceeds 2^(31 + l) by less than
// d <= 2^l, so n * m / 2^(31 + l) exceeds n / d by less than 1 / d and has its integer part. d = 1
// has l = 0, no such form: `one` passes n through.
struct FastDiv {
  unsigned m = 0, shift = 0, one = 0;
};
constexpr FastDiv fast_div(unsigned d) {
  FastDiv f;
  if (d <= 1) {
    f.one = ~0u;
    return f;
  }
  unsigned l = 0;
  while ((1ULL << l) < d) ++l;
  f.m = unsigned(((1ULL << (31 + l)) + d - 1) / d);
  f.shift = l - 1;
  return f;
}
__host__ __device__ __forceinline__ unsigned fast_quotient(unsigned n, const FastDiv &f) {
  return unsigned((unsigned long long)n * f.m >> 32 >> f.shift) + (n & f.one);
}

// Shuffle of any integer width up by `delta` lanes (wave64).
template <class T> __device__ __forceinline__ T shfl_up_any(T v, unsigned delta) {
  if constexpr (sizeof(T) == 8) return T(__shfl_up((unsigned long long)v, delta, 64));
  else return T(__shfl_up((unsigned)v, delta, 64));
}

// Mask of lanes 0..lane.
__device__ __forceinline__ unsigned long long lanes_upto(int lane) {
  return lane == 63 ? ~0ULL : ((2ULL << lane) - 1ULL);
}

// Runs of one label among a wave's 64 consecutive voxels of one x-row: every lane learns the lane
// its run starts at; a run's first lane (head) also learns the run's length. Invalid lanes are
// runs of their own. Every lane of the wave must call it.
struct WaveRun {
  bool head;
  int start_lane, len;
};
template <class T> __device__ __forceinline__ WaveRun wave_run(T l, bool valid, int x, int lane) {
  const T prev = shfl_up_any(l, 1);
  const bool start = !valid || lane == 0 || x == 0 || prev != l;
  const unsigned long long starts = __ballot(start);
  const unsigned long long after = starts & ~lanes_upto(lane);
  WaveRun r;
  r.head = start;
  r.start_lane = 63 - __clzll((long long)(starts & lanes_upto(lane)));
  r.len = (after ? __ffsll((long long)after) - 2 : 63) - lane + 1;
  return r;
}

// A workgroup's LDS table of labels (open addressing, bounded probing): run updates of one label
// fold into its slot, and the workgroup sends one global update per label it saw instead of one
// per run. A label whose probe chain is full gets -1 for good (slots are never freed), and its
// runs go to global memory directly.
constexpr int kLabelSlots = 256, kLabelProbes = 8;
struct LabelSlots {
  int tag[kLabelSlots];  // label, or -1
  __device__ void init() {
    for (int s = threadIdx.x; s < kLabelSlots; s += blockDim.x) tag[s] = -1;
  }
  static __device__ __forceinline__ int home(int l) { return int((unsigned(l) * 0x9E3779B1u) >> 24); }
  __device__ int insert(int l) {
    for (int p = 0, s = home(l); p < kLabelProbes; ++p, s = (s + 1) & (kLabelSlots - 1)) {
      const int old = atomicCAS(&tag[s], -1, l);
      if (old == -1 || old == l) return s;
    }
    return -1;
  }
  __device__ int find(int l) const {
    for (int p = 0, s = home(l); p < kLabelProbes; ++p, s = (s + 1) & (kLabelSlots - 1))
      if (tag[s] == l) return s;
    return -1;
  }
};
static_assert(kLabelSlots == 256, "home() keeps the top 8 bits of the hash");

}  // namespace brook
