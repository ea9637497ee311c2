// Field preparation per component label (batched.cu:177-255 restated for gfx950):
//   * label voxel lists (segments laid out by id, from one wave-aggregated atomic per run),
//   * one workgroup per label from a device work queue: root-search flood + argmax, DAF flood +
//     argmax (label-gated geometric SSSP, the unique float32 min-plus fixpoint), no grid barriers,
//   * the PDRF's road words and the free claim words in one streaming pass, the root rails, the target-order keys.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fields.hpp"
#include "front.hpp"
#include "tuned.hpp"

namespace brook {
namespace {

// Voxel lists: vox[seg_start[l] + slot] = every voxel of id l (slot order is free; consumers
// that need an order sort the list or reduce over it). A workgroup walks kListChunk consecutive
// voxels twice: the first pass totals each label's voxels in LDS and reserves them with one global
// add per label, the second hands out places within the reservation per x-run.
constexpr int kListChunk = 16384;

template <class CC>
__global__ void __launch_bounds__(256) fill_segments(const CC *cc, int n, Dims d, const int *seg_start, int *fill,
                                                     int *vox) {
  __shared__ LabelSlots slots;
  __shared__ int cnt[kLabelSlots], base[kLabelSlots];
  slots.init();
  for (int s = threadIdx.x; s < kLabelSlots; s += 256) cnt[s] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const long long begin = (long long)blockIdx.x * kListChunk;
  for (int t = 0; t < kListChunk; t += 256) {
    const long long g = begin + t + threadIdx.x;
    const bool valid = g < n;
    const int i = valid ? int(g) : 0;
    const CC l = valid ? cc[i] : CC(0);
    const WaveRun r = wave_run(l, valid, valid ? i % d.sx : 0, lane);
    if (!valid || l == CC(0) || !r.head) continue;
    const int s = slots.insert(int(l));
    if (s >= 0) atomicAdd(&cnt[s], r.len);
  }
  __syncthreads();
  for (int s = threadIdx.x; s < kLabelSlots; s += 256) {
    const int l = slots.tag[s];
    if (l >= 0) base[s] = atomicAdd(fill + l, cnt[s]);
    cnt[s] = 0;
  }
  __syncthreads();
  for (int t = 0; t < kListChunk; t += 256) {
    const long long g = begin + t + threadIdx.x;
    const bool valid = g < n;
    const int i = valid ? int(g) : 0;
    const CC l = valid ? cc[i] : CC(0);
    const WaveRun r = wave_run(l, valid, valid ? i % d.sx : 0, lane);
    int at = 0;
    if (valid && l != CC(0) && r.head) {
      const int s = slots.find(int(l));
      at = s >= 0 ? base[s] + atomicAdd(&cnt[s], r.len) : atomicAdd(fill + l, r.len);
    }
    at = __shfl(at, r.start_lane, 64);
    if (valid && l != CC(0)) vox[seg_start[l] + at + (lane - r.start_lane)] = i;
  }
}

// Voxel words: the neighbour mask (bit k = neighbour k of v is inside the volume and has v's nonzero
// id; every later neighbour walk reads this instead of 26 ids and bounds checks), and road words
// kFloodFree where a label is. A workgroup covers a kRecX x kRecY x kRecZ box: its ids and a one-voxel halo (0
// outside the volume, which never equals an id) are staged in LDS by coalesced row loads, the 26
// comparisons of a voxel read LDS, and each wave stores a row of 64 words of each array. Bound by
// the 12 bytes per foreground voxel and 4 per background one that it writes.
constexpr int kRecX = 64, kRecY = 4, kRecZ = 4;
template <class CC>
__global__ void __launch_bounds__(256) init_words(const CC *cc, Dims d, unsigned *mask, unsigned long long *road) {
  constexpr int TX = kRecX + 2, TY = kRecY + 2, TZ = kRecZ + 2;
  __shared__ CC tile[TZ][TY][TX];
  const int bx = int(blockIdx.x) * kRecX, by = int(blockIdx.y) * kRecY, bz = int(blockIdx.z) * kRecZ;
  for (int t = threadIdx.x; t < TX * TY * TZ; t += 256) {
    const int tx = t % TX, ty = (t / TX) % TY, tz = t / (TX * TY);
    const int x = bx + tx - 1, y = by + ty - 1, z = bz + tz - 1;
    CC v = CC(0);
    if (x >= 0 && x < d.sx && y >= 0 && y < d.sy && z >= 0 && z < d.sz)
      v = cc[x + (long long)d.sx * (y + (long long)d.sy * z)];
    tile[tz][ty][tx] = v;
  }
  __syncthreads();
  const int tx = int(threadIdx.x) % kRecX, ty = int(threadIdx.x) / kRecX;
  const int x = bx + tx, y = by + ty;
  if (x >= d.sx || y >= d.sy) return;
  for (int tz = 0; tz < kRecZ && bz + tz < d.sz; ++tz) {
    const CC l = tile[tz + 1][ty + 1][tx + 1];
    unsigned m = 0;
    if (l != CC(0)) {
      for_each_nb([&](auto K) {
        constexpr int k = decltype(K)::value;
        if (tile[tz + 1 + kDZ[k]][ty + 1 + kDY[k]][tx + 1 + kDX[k]] == l) m |= 1u << k;
      });
    }
    const long long at = x + (long long)d.sx * (y + (long long)d.sy * (bz + tz));
    mask[at] = m;
    if (l != CC(0)) road[at] = kFloodFree;
  }
}

__global__ void fill_float(float *p, long long n, float v) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

constexpr int kFloodBlock = BROOK_FLOOD_BLOCK;  // threads per label workgroup
constexpr int kFloodWaves = kFloodBlock / 64;
constexpr int kFloodPairs = BROOK_FLOOD_NB_BATCH;
// The band width is BROOK_FLOOD_BAND times the longest step.
#ifndef BROOK_FLOOD_BAND
#define BROOK_FLOOD_BAND 2.0f
#endif

// Rounds one flood of a label of `count` voxels may take (see flood_front).
__device__ __forceinline__ long long flood_budget(int count) { return 4LL * count + 4096; }

// ---- near-far bands -------------------------------------------------------------------------
// The geometric flood of a label: label-correcting rounds kept inside a distance band [.., T]. An
// improvement beyond T goes to a far list instead of the next round, and when the band has no
// front left, T moves to the nearest far distance plus the band width and the far voxels inside
// it start the next band. A voxel is then relaxed about once instead of re-queued each time a
// cheaper path with more steps arrives (30 % of pops on the 512^3 workload with anisotropy
// (8, 8, 40)). The words are the railroad's (common.hpp) with a constant cost field (all ones):
// near candidates are queued, far candidates far-listed; a near improvement of a far-listed voxel
// clears its far flag (its far entry goes stale). Far lists hold 2 * count entries (one append per
// voxel per round; a list longer than count after a round is compacted to one entry per voxel).
constexpr int kFloodFront = 4096, kFloodFar = 2048;  // entries of the lists that live in LDS
using NearList = SplitList<kFloodFront>;
using FarList = SplitList<kFloodFar>;
// n[0..2]: front lengths, rotating (round r reads n[r], appends to n[r+1], clears n[r+2]: one barrier
// per round); n[kFar0], n[kFar1]: far list lengths; n[kNone]: not appended to.
constexpr int kFar0 = 3, kFar1 = 4, kNone = 5;
constexpr int kLong = 1, kFull = 2;  // flags of a round's far list, rotating: above count, at its end
struct FloodShared {
  int n[6], flags[3];
  unsigned minfar;  // smallest far distance (float bits) since the band moved
  float T;          // the band's upper end
  int near[2][kFloodFront], far[2][kFloodFar];
  Stage stage[kFloodWaves];
};

struct FloodLists {
  NearList near[2];
  FarList far[2];
};

// Front entries b .. of one round over nc entries, at most 2P (the wave's batch): the neighbours whose
// distance they improve go to the wave's stage. W is the lane's step weight, T the band's end.
template <int P, bool Wide, class Flush>
__device__ __forceinline__ void flood_batch(const LabelTables &t, const Lane<Wide> &ln, float W, const NearList &cur, int b,
                                            int nc, unsigned T, Stage &st, int &staged, Flush &&flush) {
  int u[P];
  const int ue = batch_entries<P>(ln, cur, b, nc, u);
  unsigned long long q = 0;
  unsigned me = 0, hi[P];
  if (ln.lane < min(2 * P, nc - b)) {  // lane e: entry e's distance by the dequeue, and its mask
    q = g_or(t.road + ue, kNotQueued);
    me = g_ld(t.mask + ue);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) hi[p] = g_ld(reinterpret_cast<const unsigned *>(word_at(t.road0, ln.at(u[p]))) + 1);
  const unsigned de = road_dist(q);
  staged_pairs<P>([&](int p) {
    const unsigned m = of_entry(ln, me, 2 * p);
    const unsigned c = __float_as_uint(__uint_as_float(of_entry(ln, de, 2 * p)) + W);
    const bool later = c > T;
    const unsigned nhi = (c << 1) | unsigned(later);
    stage_put(st, staged, ((m & ln.bit) != 0u) & ((nhi | 1u) < hi[p]), u[p] + ln.off,
              ((unsigned long long)nhi << 32) | (later ? ~0u : kCostBits));
  }, flush);
}

// The staged improvements of a wave (full groups, or all of them).
__device__ __forceinline__ void flood_minima(const LabelTables &t, FloodShared &fs, Stage &st, int &staged, bool all,
                                             const NearList &nxt, int n_nxt, const FarList &far, int n_far, int count,
                                             unsigned &minfar) {
  stage_take(st, staged, all, [&](bool on, int v, unsigned long long nv) {
    unsigned long long old = 0;  // "nothing changed" unless the atomic says otherwise
    if (on) old = g_min(t.road + v, nv);
    const bool won = old > nv, later = nv & kFarListed;
    const bool near = won & !later & (int(unsigned(old)) < 0), fars = won & later & !(old & kFarListed);
    if (won & later) minfar = min(minfar, road_dist(nv));
    Appends out;
    if (!out.begin(fs.n, kNone, false, n_nxt, near, n_far, fars)) return;
    const int end = out.at[2] + out.count(2);
    const bool full = end > 2 * count;  // a wave whose appends would pass the far list's end writes none
    if (out.set[2] && end > count) atomicOr(&fs.flags[n_nxt], full ? kLong | kFull : kLong);
    if (near) nxt.put(out.place(1), v);
    if (fars & !full) far.put(out.place(2), v);
  });
}

__device__ __forceinline__ void fold_minfar(FloodShared &fs, unsigned &m) {
  if (any_lane(m != kInfBits)) {
    m = wave_min_u32(m);
    if (__lane_id() == 0) atomicMin(&fs.minfar, m);
  }
  m = kInfBits;
}

// The near list l.near[0] (fs.n[0] entries, whose words hold their start distances, queued; the other
// counters and flags 0) starts the flood. Words of the label are kFloodFree on entry but for these; on exit
// they hold the distances, every voxel dequeued. Returns false when the rounds exceed their budget
// (far above what the label-correcting rounds need: a logic error then ends as a host-visible error
// instead of a hang) or a far list its end.
template <bool Wide>
__device__ __forceinline__ bool flood_front(const LabelTables &t, const Lane<Wide> &ln, const float *W, const FloodLists &l,
                                            FloodShared &fs, int count) {
  const long long budget = flood_budget(count);
  float wmax = 0.0f;
  for (int k = 0; k < 26; ++k) wmax = fmaxf(wmax, W[k]);
  const float width = BROOK_FLOOD_BAND * wmax, weight = W[ln.k];
  Stage &st = fs.stage[ln.wave];
  NearList cur = l.near[0], nxt = l.near[1];
  FarList fcur = l.far[0], fnxt = l.far[1];
  int fc = kFar0, fn = kFar1, r = 0;
  auto swap_far = [&] {
    const FarList f = fcur; fcur = fnxt; fnxt = f;
    const int n = fc; fc = fn; fn = n;
  };
  if (threadIdx.x == 0) {
    fs.minfar = 0x7f800000u;
    fs.T = width;
  }
  __syncthreads();
  unsigned minfar = 0x7f800000u;
  long long rounds = 0;
  for (;;) {
    const unsigned T = unsigned(__builtin_amdgcn_readfirstlane(__float_as_int(fs.T)));  // moved between two barriers below
    for (;;) {             // the band's rounds
      const int nc = __builtin_amdgcn_readfirstlane(fs.n[r]);
      if (nc == 0) break;
      if (++rounds > budget) return false;  // uniform
      const int rn = rot_next(r);
      if (threadIdx.x == 0) fs.n[rot_prev(r)] = fs.flags[rot_prev(r)] = 0;
      int staged = 0;
      with_pairs<kFloodPairs>(nc, kFloodWaves, [&](auto Pairs) {
        constexpr int P = decltype(Pairs)::value;
        for (int b = ln.wave * 2 * P; b < nc; b += kFloodWaves * 2 * P)
          flood_batch<P>(t, ln, weight, cur, b, nc, T, st, staged,
                         [&] { flood_minima(t, fs, st, staged, false, nxt, rn, fcur, fc, count, minfar); });
      });
      flood_minima(t, fs, st, staged, true, nxt, rn, fcur, fc, count, minfar);
      fold_minfar(fs, minfar);
      __syncthreads();
      r = rn;
      const NearList f = cur; cur = nxt; nxt = f;
      const int flags = fs.flags[r];
      if (flags & kFull) return false;
      if (flags & kLong) {  // one entry per far-listed voxel (the one whose atomic clears its far flag)
        const int nf = fs.n[fc];
        for (int i = threadIdx.x; i < nf; i += blockDim.x) {
          const int w = fcur.get(i);
          if (g_and(t.road + w, ~kFarListed) & kFarListed) fnxt.put(wave_slot(&fs.n[fn]), w);
        }
        __syncthreads();
        const int kept = fs.n[fn];
        for (int i = threadIdx.x; i < kept; i += blockDim.x) g_or(t.road + fnxt.get(i), kFarListed);
        if (threadIdx.x == 0) fs.n[fc] = 0;
        __syncthreads();
        swap_far();
      }
    }
    const int nf = fs.n[fc];
    if (nf == 0) return true;
    if (++rounds > budget) return false;
    const float next = __uint_as_float(fs.minfar) + width;  // the band moves to the nearest far distance
    __syncthreads();
    if (threadIdx.x == 0) {
      fs.T = next;
      fs.minfar = 0x7f800000u;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nf; i += blockDim.x) {  // far voxels inside the band start it
      const int w = fcur.get(i);
      if (!(lp_u64(t.road + w) & kFarListed)) continue;
      const unsigned long long was = g_and(t.road + w, ~(kFarListed | kNotQueued));
      if (!(was & kFarListed)) continue;
      if (__uint_as_float(road_dist(was)) <= next) {
        cur.put(wave_slot(&fs.n[r]), w);
      } else {
        g_or(t.road + w, kFarListed | kNotQueued);
        minfar = min(minfar, road_dist(was));
        fnxt.put(wave_slot(&fs.n[fn]), w);
      }
    }
    fold_minfar(fs, minfar);
    __syncthreads();
    if (threadIdx.x == 0) fs.n[fc] = 0;  // appended to again after two more barriers
    swap_far();
  }
}

__device__ __forceinline__ void flood_clear(FloodShared &fs) {
  if (threadIdx.x < 6) fs.n[threadIdx.x] = 0;
  if (threadIdx.x < 3) fs.flags[threadIdx.x] = 0;
}

template <bool Wide>
__device__ __forceinline__ bool flood_label(const LabelTables &t, const Lane<Wide> &ln, int src, const float *W,
                                            const FloodLists &l, FloodShared &fs, int count) {
  flood_clear(fs);
  __syncthreads();
  if (threadIdx.x == 0) {
    sp_u64(t.road + src, road_word(0u, 0ULL, kCostBits));  // distance 0, queued
    l.near[0].put(0, src);
    fs.n[0] = 1;
  }
  __syncthreads();
  return flood_front(t, ln, W, l, fs, count);
}

// The free-space length of a soma voxel at offset (dxi, dyi, dzi) from the root, when its physical
// distance is within `radius`: the shortest 26-connected path through empty space, in float32 in
// the order of freespace_seed_lab (batched_regular.inc:51-73).
__device__ __forceinline__ bool free_space(int dxi, int dyi, int dzi, float wx, float wy, float wz, float radius, float &val) {
  const float rdx = wx * (float)dxi, rdy = wy * (float)dyi, rdz = wz * (float)dzi;
  if (rdx * rdx + rdy * rdy + rdz * rdz > radius * radius) return false;
  const float dx = fabsf((float)dxi), dy = fabsf((float)dyi), dz = fabsf((float)dzi);
  const float dxyz = fminf(fminf(dx, dy), dz);
  const float dxy = fminf(dx, dy), dyz = fminf(dy, dz), dxz = fminf(dx, dz);
  val = dxyz * sqrtf(wx * wx + wy * wy + wz * wz) + wx * (dx - dxyz) + wy * (dy - dxyz) + wz * (dz - dxyz) +
        (dxy - dxyz) * (sqrtf(wx * wx + wy * wy) - wx - wy) + (dxz - dxyz) * (sqrtf(wx * wx + wz * wz) - wx - wz) +
        (dyz - dxyz) * (sqrtf(wy * wy + wz * wz) - wy - wz);
  return true;
}

// A soma's DAF flood (batched.cu:222-231): every voxel of the label inside the free-space ball
// starts at its free-space length (the root at 0), then the label-correcting rounds.
template <bool Wide>
__device__ __forceinline__ bool flood_free_space(const LabelTables &t, Dims d, const Lane<Wide> &ln, const int *list, int cnt, int root,
                                                 float radius, const float *W, const FloodLists &l, FloodShared &fs) {
  flood_clear(fs);
  __syncthreads();
  int rx, ry, rz;
  unravel(root, d, rx, ry, rz);
  for (int j = threadIdx.x; j < cnt; j += blockDim.x) {
    const int v = g_ld(list + j);
    int x, y, z;
    unravel(v, d, x, y, z);
    float val;
    if (!free_space(x - rx, y - ry, z - rz, W[0], W[2], W[4], radius, val)) continue;
    sp_u64(t.road + v, road_word(__float_as_uint(val), 0ULL, kCostBits));  // queued
    l.near[0].put(wave_slot(&fs.n[0]), v);
  }
  __syncthreads();
  return flood_front(t, ln, W, l, fs, cnt);
}

// Argmax of the flooded distance over the label's voxel list: largest finite value, ties -> lowest
// flat index (the packed key of batched_regular.inc:9-22). Returns the key (0: none).
__device__ __forceinline__ unsigned long long label_argmax(const unsigned long long *road, const int *list, int count,
                                                           unsigned long long *lds) {
  if (threadIdx.x == 0) *lds = 0;
  __syncthreads();
  unsigned long long best = 0;
  for (int j = threadIdx.x; j < count; j += blockDim.x) {
    int v = g_ld(list + j);
    const unsigned fb = road_dist(lp_u64(road + v));  // unreached: +inf
    if (!(fb < 0x7f800000u)) continue;
    unsigned long long key = ((unsigned long long)fb << 32) | (unsigned long long)(0xFFFFFFFFu - (unsigned)v);
    best = key > best ? key : best;
  }
  for (int off = 32; off > 0; off >>= 1) {
    unsigned long long o = __shfl_down(best, off, 64);
    best = o > best ? o : best;
  }
  if ((threadIdx.x & 63) == 0 && best) atomicMax(lds, best);
  __syncthreads();
  unsigned long long r = *lds;
  __syncthreads();
  return r;
}

// stalled: set when a flood exceeded its round budget (the label's fields are then left as they
// are and the host raises). The queue is sorted largest first: workgroup w < nfixed (resident from
// the start, at most the queue's length) takes item w first (workgroups go to the XCDs in turn, so
// the largest labels start on different XCDs); every other item comes from the shared cursor,
// from item nfixed on.
template <bool Wide>
__global__ void __launch_bounds__(kFloodBlock) prepare_labels(const FloodJob *__restrict__ jobs,
                                                              const int2 *__restrict__ queue, int nqueue, int nfixed,
                                                              int *next, int *stalled) {
  __shared__ float W[26];
  __shared__ FloodShared fs;
  __shared__ unsigned long long best;
  __shared__ int item;
  for (bool first_item = true;; first_item = false) {
    __syncthreads();
    if (threadIdx.x == 0) item = first_item && int(blockIdx.x) < nfixed ? int(blockIdx.x) : nfixed + atomicAdd(next, 1);
    __syncthreads();
    if (item >= nqueue) return;
    const int2 q = queue[item];
    const FloodJob job = jobs[__builtin_amdgcn_readfirstlane(q.x)];  // uniform: scalar registers
    const int L = __builtin_amdgcn_readfirstlane(q.y);
    const Dims d = job.d;
    const LabelTables &t = job.t;
    if (threadIdx.x < 26) W[threadIdx.x] = g_ld(t.weights + threadIdx.x);
    const Lane<Wide> ln = lane_of<Wide>(d);
    __syncthreads();
    const int s0 = __builtin_amdgcn_readfirstlane(g_ld(t.seg_start + L));  // uniform: scalar registers
    const int cnt = __builtin_amdgcn_readfirstlane(g_ld(t.seg_count + L));
    const int *list = t.vox + s0;
    const FloodLists lists{{NearList{job.lists_a + s0, fs.near[0]}, NearList{job.lists_b + s0, fs.near[1]}},
                           {FarList{job.far_a + 2LL * s0, fs.far[0]}, FarList{job.far_b + 2LL * s0, fs.far[1]}}};
    long long root = g_ld(t.root + L);
    if (root < 0) {  // no border target: flood from the component's first voxel, root = argmax
      if (!flood_label(t, ln, int(g_ld(t.first + L)), W, lists, fs, cnt)) {
        if (threadIdx.x == 0) atomicOr(stalled, 1);
        continue;
      }
      unsigned long long key = label_argmax(t.road, list, cnt, &best);
      root = key ? (long long)(0xFFFFFFFFu - (unsigned)key) : -1;
      for (int j = threadIdx.x; j < cnt; j += blockDim.x) sp_u64(t.road + g_ld(list + j), kFloodFree);
      __syncthreads();
      if (threadIdx.x == 0) g_st(t.root + L, root);
      if (job.root_only) continue;
    }
    const float radius = t.free_radius ? g_ld(t.free_radius + L) : 0.0f;
    const bool converged = radius > 0.0f ? flood_free_space(t, d, ln, list, cnt, int(root), radius, W, lists, fs)
                                         : flood_label(t, ln, int(root), W, lists, fs, cnt);
    if (!converged) {
      if (threadIdx.x == 0) atomicOr(stalled, 1);
      continue;
    }
    unsigned long long key = label_argmax(t.road, list, cnt, &best);
    if (threadIdx.x == 0) {
      g_st(t.target + L, key ? (long long)(0xFFFFFFFFu - (unsigned)key) : -1LL);
      g_st(t.max_daf + L, key ? __uint_as_float((unsigned)(key >> 32)) : 0.0f);
    }
    for (int j = threadIdx.x; j < cnt; j += blockDim.x) {  // DAF out, words back to kFloodFree
      const int v = g_ld(list + j);
      g_st(job.daf + v, __uint_as_float(road_dist(lp_u64(t.road + v))));
      sp_u64(t.road + v, kFloodFree);
    }
  }
}

// PDRF (batched_regular.inc:93-108), the road word that carries it and the claim word (alive) in one
// pass. use[l] 0: not traced.
template <class CC>
__global__ void __launch_bounds__(256) pdrf_alive(const CC *cc, const float *dbf, const float *daf, const float *M,
                                                  const float *inv, const unsigned char *use, int squarings, float scale,
                                                  long long n, float *pdrf, unsigned long long *road,
                                                  unsigned long long *claim) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  CC l = cc[i];
  unsigned char u = use[l];
  if (l == CC(0) || u == 0) {
    if (pdrf) pdrf[i] = kInf;
    return;
  }
  float dv = dbf[i];
  if (dv == 0.0f) dv = kInf;
  float p = 1.0f - dv * M[l];
  for (int k = 0; k < squarings; ++k) p = p * p;
  p = p * scale;
  if (u == 2) {
    float a = daf[i];
    if (isinf(a)) a = 0.0f;
    p = p + a * inv[l];
  }
  if (pdrf) pdrf[i] = p;
  road[i] = kUnreached | (__float_as_uint(p) & kCostBits);
  claim[i] = kFree;
}

__global__ void set_rails(unsigned long long *road, const long long *root, const int *labels, int count) {
  int i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) road[root[labels[i]]] = kUnreached;
}

unsigned grid_for(long long n) { return unsigned((n + 255) / 256); }
unsigned blocks_of(long long n, int per) { return unsigned((n + per - 1) / per); }

}  // namespace

void build_segments(Context &ctx, const void *cc, int cc_bytes, Dims d, const std::vector<int> &seg_start,
                    Buffer<int> &seg_start_dev, Buffer<int> &vox) {
  const int n = d.sx * d.sy * d.sz;
  seg_start_dev = Buffer<int>(ctx, seg_start.size());
  seg_start_dev.upload(ctx, seg_start.data(), seg_start.size());
  Buffer<int> fill(ctx, seg_start.size());
  fill.clear(ctx);
  vox = Buffer<int>(ctx, std::max(1, seg_start.back()));
  if (cc_bytes == 1)
    fill_segments<uint8_t><<<blocks_of(n, kListChunk), 256, 0, ctx.stream()>>>(static_cast<const uint8_t *>(cc), n, d,
                                                                  seg_start_dev.data(), fill.data(), vox.data());
  else if (cc_bytes == 2)
    fill_segments<uint16_t><<<blocks_of(n, kListChunk), 256, 0, ctx.stream()>>>(static_cast<const uint16_t *>(cc), n, d,
                                                                   seg_start_dev.data(), fill.data(), vox.data());
  else
    fill_segments<uint32_t><<<blocks_of(n, kListChunk), 256, 0, ctx.stream()>>>(static_cast<const uint32_t *>(cc), n, d,
                                                                   seg_start_dev.data(), fill.data(), vox.data());
  BROOK_LAUNCHED();
}

void voxel_words(Context &ctx, const void *cc, int cc_bytes, Dims d, unsigned *mask, unsigned long long *road) {
  const long long n = (long long)d.sx * d.sy * d.sz;
  if (n == 0) return;
  KernelTimer kt(ctx, "init_words");
  if ((d.sy + kRecY - 1) / kRecY > 65535 || (d.sz + kRecZ - 1) / kRecZ > 65535)
    throw std::invalid_argument("volume too tall for the record tiles");
  const dim3 g(unsigned((d.sx + kRecX - 1) / kRecX), unsigned((d.sy + kRecY - 1) / kRecY), unsigned((d.sz + kRecZ - 1) / kRecZ));
  if (cc_bytes == 1)
    init_words<uint8_t><<<g, 256, 0, ctx.stream()>>>(static_cast<const uint8_t *>(cc), d, mask, road);
  else if (cc_bytes == 2)
    init_words<uint16_t><<<g, 256, 0, ctx.stream()>>>(static_cast<const uint16_t *>(cc), d, mask, road);
  else
    init_words<uint32_t><<<g, 256, 0, ctx.stream()>>>(static_cast<const uint32_t *>(cc), d, mask, road);
  BROOK_LAUNCHED();
}

void fill_value(Context &ctx, float *p, long long n, float v) {
  if (n <= 0) return;
  fill_float<<<grid_for(n), 256, 0, ctx.stream()>>>(p, n, v);
  BROOK_LAUNCHED();
}

void prepare_fields(Context &ctx, const std::vector<FloodJob> &jobs, const std::vector<LabelItem> &items, int max_grid) {
  if (items.empty()) return;
  Buffer<FloodJob> jobs_dev(ctx, jobs.size());
  jobs_dev.upload(ctx, jobs.data(), jobs.size());
  std::vector<int2> q(items.size());
  for (size_t i = 0; i < items.size(); ++i) q[i] = make_int2(items[i].sample, items[i].label);
  Buffer<int2> queue(ctx, q.size());
  queue.upload(ctx, q.data(), q.size());
  Buffer<int> next(ctx, 2);  // [0] queue cursor, [1] stalled
  next.clear(ctx);
  const int nq = int(q.size());
  bool wide = false;  // one launch serves every sample of the group
  for (const FloodJob &j : jobs) wide |= !narrow_words(j.d);
  // every workgroup takes labels from the queue until it is spent, so any grid drains it
  int grid = std::min(nq, BROOK_FLOOD_GRID > 0 ? BROOK_FLOOD_GRID : ctx.compute_units() * 2);
  if (max_grid > 0) grid = std::min(grid, max_grid);
  {
    KernelTimer kt(ctx, "prepare_labels");
    (wide ? prepare_labels<true> : prepare_labels<false>)<<<grid, kFloodBlock, 0, ctx.stream()>>>(jobs_dev.data(), queue.data(), nq,
                                                           std::min(grid, ctx.compute_units()), next.data(),
                                                           next.data() + 1);
    BROOK_LAUNCHED();
  }
  if (next.download(ctx)[1]) throw std::runtime_error("flood did not converge: a label exceeded its round budget");
}

void pdrf_and_alive(Context &ctx, const void *cc, int cc_bytes, long long n, const float *dbf, const float *daf,
                    const float *M, const float *inv, const unsigned char *use, int squarings, float scale, float *pdrf,
                    unsigned long long *road, unsigned long long *claim) {
  KernelTimer kt(ctx, "pdrf_alive");
  if (cc_bytes == 1)
    pdrf_alive<uint8_t><<<grid_for(n), 256, 0, ctx.stream()>>>(static_cast<const uint8_t *>(cc), dbf, daf, M, inv, use,
                                                               squarings, scale, n, pdrf, road,
                                                               claim);
  else if (cc_bytes == 2)
    pdrf_alive<uint16_t><<<grid_for(n), 256, 0, ctx.stream()>>>(static_cast<const uint16_t *>(cc), dbf, daf, M, inv, use,
                                                                squarings, scale, n, pdrf, road,
                                                               claim);
  else
    pdrf_alive<uint32_t><<<grid_for(n), 256, 0, ctx.stream()>>>(static_cast<const uint32_t *>(cc), dbf, daf, M, inv, use,
                                                                squarings, scale, n, pdrf, road,
                                                               claim);
  BROOK_LAUNCHED();
}

void root_rails(Context &ctx, unsigned long long *road, const long long *root, const int *labels, int count) {
  if (!count) return;
  set_rails<<<grid_for(count), 256, 0, ctx.stream()>>>(road, root, labels, count);
  BROOK_LAUNCHED();
}

}  // namespace brook
