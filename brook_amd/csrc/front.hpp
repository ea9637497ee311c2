// Frontier machinery of the label workgroups (floods, railroad, invalidation): a front entry's 26
// neighbours are served by the 32 lanes of half a wave, one neighbour per lane.
//
// What bounds a round. A front's neighbour words are scattered 8-byte accesses, 9 rows of 3 per
// entry, and a compute unit takes about one cache line per cycle: lanes are therefore in address
// order (x fastest), so the three lanes of a row read one 24-byte piece and an entry costs 9 to 11
// lines where a thread per entry costs 26. The other limit is instruction issue (a vector
// instruction of a wave takes its SIMD four cycles): with a neighbour per lane the list appends are
// ballots instead of wave scans, addresses are a 32-bit offset on a scalar base, the words are padded so
// that no address is clamped, and what only depends on the entry is computed once, in the lane that
// holds the entry, and passed to its half by one LDS permute. Neighbour words are loaded beside the
// entry's own mask and dequeue, not after them, so a round is two dependent memory steps: loads,
// then atomic minima.
#pragma once
#include "common.hpp"

namespace brook {

// The neighbour table's index of each lane slot: slots 0..25 are the 26 neighbours by ascending
// (z, y, x), i.e. ascending address.
struct SlotTable {
  int k[26];
};
constexpr SlotTable slot_table() {
  SlotTable t{};
  for (int k = 0; k < 26; ++k) {
    int before = 0;
    for (int j = 0; j < 26; ++j) {
      const int a = (kDZ[j] + 1) * 9 + (kDY[j] + 1) * 3 + kDX[j] + 1, b = (kDZ[k] + 1) * 9 + (kDY[k] + 1) * 3 + kDX[k] + 1;
      before += a < b;
    }
    t.k[before] = k;
  }
  return t;
}
__constant__ static const SlotTable kSlots = slot_table();

// A thread's place: half a wave (32 lanes) per entry, lane slot s of a half for neighbour slot s;
// slots 26..31 are the entry itself (kCentre for walks that read it too) and test no mask bit.
// Off: byte offsets into the padded word arrays (narrow_words: 32 bits).
constexpr int kCentre = 26;
template <bool Wide> struct Lane {
  using Off = std::conditional_t<Wide, unsigned long long, unsigned>;
  int lane, half, wave;  // lane in the wave, which half, wave in the workgroup
  int slot, k, off;      // slot, its neighbour and flat offset
  unsigned bit;          // the neighbour's mask bit (0: slot of the entry itself)
  Off offb;              // (off + pad) * 8
  float dx, dy, dz;
  __device__ __forceinline__ Off at(int u) const { return (Off(unsigned(u)) << 3) + offb; }
};
template <bool Wide> __device__ __forceinline__ Lane<Wide> lane_of(const Dims &d) {
  Lane<Wide> l;
  l.lane = int(threadIdx.x) & 63;
  l.half = l.lane >> 5;
  l.wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  l.slot = l.lane & 31;
  const bool nb = l.slot < 26;
  l.k = nb ? kSlots.k[l.slot] : 0;
  const int dx = nb ? kNX[l.k] : 0, dy = nb ? kNY[l.k] : 0, dz = nb ? kNZ[l.k] : 0;
  l.off = step_offset(d, dx, dy, dz);
  l.bit = nb ? 1u << l.k : 0u;
  l.offb = typename Lane<Wide>::Off((l.off + word_pad(d)) * 8);
  l.dx = float(dx);
  l.dy = float(dy);
  l.dz = float(dz);
  return l;
}
// The padded word at a byte offset from the array's first pad word.
template <class Off> __device__ __forceinline__ unsigned long long *word_at(unsigned long long *first, Off off) {
  return reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(first) + off);
}

__device__ __forceinline__ unsigned long long ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ bool any_lane(bool b) { return ballot(b) != 0; }
// Value v of lane 2p + half (the entry of the caller's half in pair p).
template <class L> __device__ __forceinline__ unsigned of_entry(const L &ln, unsigned v, int from) {
  return unsigned(__builtin_amdgcn_ds_bpermute((from + ln.half) << 2, int(v)));
}
template <class L> __device__ __forceinline__ float of_entry(const L &ln, float v, int from) {
  return __uint_as_float(of_entry(ln, __float_as_uint(v), from));
}

// ---- reductions over rows of 16 lanes, halves and waves (all lanes active) ----------------------
template <int Ctrl> __device__ __forceinline__ unsigned dpp(unsigned v) {
  return unsigned(__builtin_amdgcn_update_dpp(int(v), int(v), Ctrl, 0xF, 0xF, false));
}
// Minimum over the lane's half (32 lanes): four steps inside a row (xor 1, xor 2, mirrored halves,
// mirrored row), then the other row.
__device__ __forceinline__ unsigned half_min(unsigned v) {
  v = min(v, dpp<0xB1>(v));
  v = min(v, dpp<0x4E>(v));
  v = min(v, dpp<0x141>(v));
  v = min(v, dpp<0x140>(v));
  return min(v, unsigned(__builtin_amdgcn_ds_swizzle(int(v), 0x401F)));  // lane ^ 16
}
__device__ __forceinline__ unsigned long long half_min_u64(unsigned long long v) {
  const unsigned hi = unsigned(v >> 32), h = half_min(hi);
  const unsigned lo = half_min(hi == h ? unsigned(v) : ~0u);
  return ((unsigned long long)h << 32) | lo;
}
__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
  v = half_min(v);
  return min(unsigned(__builtin_amdgcn_readlane(int(v), 0)), unsigned(__builtin_amdgcn_readlane(int(v), 32)));
}
__device__ __forceinline__ unsigned long long wave_least(unsigned long long v) {
  const unsigned hi = unsigned(v >> 32), h = wave_min_u32(hi);
  const unsigned lo = wave_min_u32(hi == h ? unsigned(v) : ~0u);
  return ((unsigned long long)h << 32) | lo;
}

// Set bits of m below this lane.
__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return int(__builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0u)));
}

// Pairs of entries (one per half) a wave has in flight in a round of n entries, with `waves` waves:
// the least of 1, 2, 4, Max that serves the front in one batch per wave, so that a small front
// spreads over all waves; longer fronts take several batches of Max.
template <int Max, class F> __device__ __forceinline__ void with_pairs(int n, int waves, F &&f) {
  using std::integral_constant;
  if (n <= 2 * waves) f(integral_constant<int, 1>{});
  else if (n <= 4 * waves) f(integral_constant<int, 2>{});
  else if (Max <= 4 || n <= 8 * waves) f(integral_constant<int, 4>{});
  else f(integral_constant<int, Max>{});
}

// A wave's candidates for the atomic minima. An atomic instruction of a wave costs about 37 ns whether 18
// or 52 of its lanes are active (512^3 workload's pattern, 16 waves on a compute unit; the load of
// the same words 8 ns per entry), and only about a quarter of an entry's neighbours pass the check
// against the loaded words. So the lanes that pass write (voxel, word) to the wave's stage in LDS, and
// the minima and everything that follows from their old words run on full groups of 64. Room for
// what may be left and kStagePairs pairs' neighbours.
constexpr int kStagePairs = 3;
constexpr int kStage = 64 + 2 * kStagePairs * 26;
struct Stage {
  unsigned long long word[kStage];
  int voxel[kStage];
};
// LDS written by other lanes of the wave: the wave's LDS operations complete in order, so only the
// compiler has to keep them.
__device__ __forceinline__ void stage_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// Stages the lanes with `on`; n is the wave's count. All lanes active.
__device__ __forceinline__ void stage_put(Stage &st, int &n, bool on, int voxel, unsigned long long word) {
  const unsigned long long m = ballot(on);
  if (on) {
    const int at = n + lanes_below(m);
    st.word[at] = word;
    st.voxel[at] = voxel;
  }
  n += __popcll(m);
}
// Calls pair(p) for each of P pairs and flush() after every kStagePairs of them.
template <int P, class F, class G> __device__ __forceinline__ void staged_pairs(F &&pair, G &&flush) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
    pair(p);
    if (p % kStagePairs == kStagePairs - 1 || p == P - 1) flush();
  }
}
// Calls group(lane is on, voxel, word) on the last 64 staged entries while there are that many, and
// with `all` on what is left.
template <class F> __device__ __forceinline__ void stage_take(Stage &st, int &n, bool all, F &&group) {
  const int lane = __lane_id();
  while (n >= 64 || (all && n > 0)) {
    stage_fence();
    const int from = n >= 64 ? n - 64 : 0;
    const bool on = lane < n - from;
    const int at = from + (on ? lane : 0);
    const int voxel = st.voxel[at];
    const unsigned long long word = st.word[at];
    n = from;
    group(on, voxel, word);
    stage_fence();
  }
}

// Appends of one wave to up to three lists whose lengths are LDS counters n[i0], n[i1], n[i2]: one
// LDS add per list with entries (three lanes of one instruction), then the lanes' places. All lanes
// active.
struct Appends {
  unsigned long long set[3];
  int at[3];
  // false: nothing to append
  __device__ __forceinline__ bool begin(int *n, int i0, bool a, int i1, bool b, int i2, bool c) {
    set[0] = ballot(a);
    set[1] = ballot(b);
    set[2] = ballot(c);
    if (!(set[0] | set[1] | set[2])) return false;
    const int lane = __lane_id();
    const int add = lane == 0 ? __popcll(set[0]) : lane == 1 ? __popcll(set[1]) : __popcll(set[2]);
    int base = 0;
    if (lane < 3 && add) base = atomicAdd(n + (lane == 0 ? i0 : lane == 1 ? i1 : i2), add);
    for (int j = 0; j < 3; ++j) at[j] = __builtin_amdgcn_readlane(base, j);
    return true;
  }
  __device__ __forceinline__ int count(int j) const { return __popcll(set[j]); }
  __device__ __forceinline__ int place(int j) const { return at[j] + lanes_below(set[j]); }
};

// Rotation over three counters (see the rounds).
__device__ __forceinline__ int rot_next(int r) { return r == 2 ? 0 : r + 1; }
__device__ __forceinline__ int rot_prev(int r) { return r == 0 ? 2 : r - 1; }

// A list of a label workgroup: entry j in LDS below N, in the label's device list beyond, so that the
// appends and reads of a short list never wait for device memory.
template <int N> struct SplitList {
  int *g;
  int *s;
  __device__ __forceinline__ int get(int j) const { return j < N ? s[j] : lp_i(g + j); }
  __device__ __forceinline__ void put(int j, int v) const {
    if (j < N) s[j] = v;
    else g_st(g + j, v);
  }
  // get() of entries that all lie below `length`.
  __device__ __forceinline__ int get(int j, int length) const { return length <= N ? s[j] : get(j); }
};

// Entries b .. b + n - 1 of a list of `length` entries (1 <= n <= 2P, b + n <= length): lane e holds
// entry e (lanes >= n the last one), u[p] is the entry of the lane's half in pair p.
template <int P, class L, class List>
__device__ __forceinline__ int batch_entries(const L &ln, const List &list, int b, int length, int (&u)[P]) {
  const int last = length - 1;
#pragma unroll
  for (int p = 0; p < P; ++p) u[p] = list.get(min(b + 2 * p + ln.half, last), length);
  return list.get(min(b + ln.lane, last), length);
}

}  // namespace brook
