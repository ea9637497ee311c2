// The TEASAR trace loop on gfx950: one workgroup per component label, labels pulled from a
// device work queue (largest first), every label's whole path sequence traced inside its
// workgroup with workgroup barriers only -- no grid-wide barrier, no host round trip per path.
//
// Per label, exactly the semantics of the reference's lockstep tracer (labels never interact, so
// one label at a time is exact; lockstep.cu:91-622, lockstep_coop.inc, lockstep_regular.inc):
//   target     manual targets first (in pop order), then the first alive voxel of the label's
//              descending-DAF order at or after its cursor          (lockstep_coop.inc:343-416)
//   railroad   vertex-weighted SSSP from the target with the one-ulp step, rails absorb, near-far
//              bands bounded by the best rail; the stop rail is min (distance, flat index)
//                                                                   (lockstep_coop.inc:71-305)
//   backtrace  one wave: lane k probes neighbour k, two wave-min reductions give the lowest k
//              among the smallest distances; the join takes u's first rail in dijkstra3d order
//                                                                   (lockstep_regular.inc:61-154)
//   rails      path voxels get PDRF 0                               (lockstep_regular.inc:246-251)
//   invalidate rolling ball, bands of the bottleneck M on a fixed grid, synchronous rounds from
//              a snapshot inside a band, exact pulls at band boundaries
//                                                         (invalidation_kernels.cuh:105-299)
// Neighbour walks read the per-voxel same-label mask (one word instead of 26 ids), and half a wave
// serves a front entry, a lane per neighbour (front.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "front.hpp"
#include "trace.hpp"
#include "tuned.hpp"

namespace brook {
namespace {

constexpr int kBlock = BROOK_TRACE_BLOCK;  // threads per label workgroup
constexpr int kWaves = kBlock / 64;
constexpr int kMaxPairs = BROOK_NB_BATCH;
constexpr unsigned long long kMinfarNone = 0x7f8000007f800000ULL;
constexpr int kProf = kTraceProfileSlots;
// A railroad band's width in costs of its first voxel. Narrow bands relax a voxel less often, wide
// ones take fewer rounds. Slowest label of the 512^3 workload, railroads in ms (entries relaxed):
// width 4 54.9 (1.65 M), 2 35.7 (936 k), 1 31.0 (696 k), 0.5 30.6 (523 k); a 48-voxel crop of three
// tubes 1.73, 1.76, 1.80, 2.02; a 31 M voxel request 9.4, 7.0, 6.6, 6.9.
#ifndef BROOK_ROAD_BAND
#define BROOK_ROAD_BAND 1.0f
#endif

// Entries of the near fronts and of the far (waiting) lists that live in LDS; longer lists go on in
// the label's device memory. (Registers allow one workgroup of 1024 threads per compute unit, so the
// workgroup may take most of its 160 KB.)
constexpr int kLdsFront = 3072, kLdsFar = 2048;
constexpr int kRadiusSlots = 4096;
using Front = SplitList<kLdsFront>;
using Far = SplitList<kLdsFar>;

// List lengths (Shared::n). Front lengths rotate over three counters: round r reads n[r], appends to
// n[r+1] and clears n[r+2] (read in round r-1), so a round needs one barrier. Waves leave the rounds by
// reading n[r] = 0, so a barrier comes before the next append to n[r] (a band's promotions). The far
// (waiting) lengths rotate likewise over kFar .. kFar + 2, a step per phase (band).
constexpr int kFar = 3, kTouched = 6, kStale = 7, kDirty = 8, kCounters = 9;

// What a round found about the railroad's far list, in the rotation of the front lengths (a wave
// ahead by a barrier writes another slot than the one its workgroup still reads): kLong, more than
// `count` entries (compacted); kFull, an append found the list at its end (never expected).
constexpr int kLong = 1, kFull = 2;

struct Shared {
  int n[kCounters], flags[3];
  int done, target, path_len, found;
  long long cursor, seg_end;
  int pcount, ordered, after_used;  // ordered: the current target came from the DAF order
  unsigned lowest[3];               // invalidation: least waiting bottleneck, rotating per band
  float T;
  unsigned long long rail_best, minfar;
  int store_pos;
  // per-label profile: [0] total [1] target [2] railroad [3] backtrace [4] invalidation (wall-clock
  // ticks), [5] railroad rounds, [6] invalidation rounds, [7] paths, [8] railroad phases,
  // [9] far entries scanned, [10] near entries expanded, [11] invalidation entries expanded,
  // [12] waiting entries scanned, [13] bands, [14] entries pulled
  unsigned long long prof[kProf];
  long long tick;
  int front[2][kLdsFront];
  int far[2][kLdsFar];
  // invalidation: ball radii of the path's voxels by source (see source_radius)
  unsigned long long radius[kRadiusSlots];
  Stage stage[kWaves];
};

// A label's lists: near fronts, far lists (the far device lists hold two entries per voxel), and the
// invalidation's scratch (two ints, or one snapshot, per voxel each).
struct Lists {
  Front near[2];
  Far far[2];
  int *touched, *walk;
  unsigned long long *snap;
  int *stale;
};
__device__ __forceinline__ Lists lists_of(const TraceArgs &a, Shared &sh, int seg) {
  return Lists{{Front{a.lists[0] + seg, sh.front[0]}, Front{a.lists[1] + seg, sh.front[1]}},
               {Far{a.lists[2] + 2LL * seg, sh.far[0]}, Far{a.lists[3] + 2LL * seg, sh.far[1]}},
               a.lists[4] + seg, a.lists[5] + seg, a.snaps[0] + seg, reinterpret_cast<int *>(a.snaps[1] + seg)};
}

// Rounds (and phases) one railroad or invalidation may take before the label is given up as not
// converging: far above what the label-correcting rounds need (a few per voxel of the label at
// most), and finite, so a logic error ends as a host-visible error instead of a hang.
__device__ __forceinline__ long long round_budget(int count) { return 4LL * count + 4096; }

// Statuses of one railroad: 1 nearest rail settled, 2 no rail reachable, 3 did not converge
// within the round budget, 4 a far list overflowed.
constexpr int kRailFound = 1, kNoRail = 2, kStalled = 3, kOverflowed = 4;
// counters[8] bits: 1 = a railroad or invalidation did not converge, 2 = a far list overflowed.
__device__ __forceinline__ void report_failure(const TraceArgs &a, int status) {
  g_or(a.counters + 8, status == kStalled ? 1 : 2);
}

__device__ __forceinline__ void lap(Shared &sh, int slot) {
  if (threadIdx.x == 0) {
    long long now = wall_clock64();
    sh.prof[slot] += (unsigned long long)(now - sh.tick);
    sh.tick = now;
  }
}

__device__ __forceinline__ unsigned mask_of(const TraceArgs &a, int v) { return g_ld(a.mask + v); }
// The neighbours v may pull from (see TraceArgs::inmask).
__device__ __forceinline__ unsigned in_mask(const TraceArgs &a, int v) {
  return a.inmask ? g_ld(a.inmask + v) : mask_of(a, v);
}
// Voxel coordinates by high products instead of divisions.
__device__ __forceinline__ void place(const TraceArgs &a, int v, int &x, int &y, int &z) {
  z = int(fast_quotient(unsigned(v), a.by_plane));
  const int r = v - z * (a.d.sx * a.d.sy);
  y = int(fast_quotient(unsigned(r), a.by_row));
  x = r - y * a.d.sx;
}

// ---- railroad -------------------------------------------------------------------------------
// Distances live in the road words (common.hpp). A front voxel is dequeued by one atomic or that
// also returns its distance; an improvement is one atomic minimum whose old value says whether the
// voxel still has to be queued or far-listed. Near candidates are queued (no flag), rails not queued,
// far candidates far-listed and not queued; a near improvement of a far-listed voxel clears its far
// flag, so its far-list entry goes stale. A rail is recognised by its zero cost.
// Per-thread minima of the reached rails and far distances are folded into LDS once per round.
struct RoadMins {
  unsigned long long rail = kMaxKey, far = kMinfarNone;
};

__device__ __forceinline__ void road_fold(Shared &sh, RoadMins &mins) {
  if (any_lane(mins.rail != kMaxKey)) {
    const unsigned long long r = wave_least(mins.rail);
    if (__lane_id() == 0) atomicMin(&sh.rail_best, r);
  }
  if (any_lane(mins.far != kMinfarNone)) {
    const unsigned long long f = wave_least(mins.far);
    if (__lane_id() == 0) atomicMin(&sh.minfar, f);
  }
  mins = RoadMins{};
}

// The lists of a railroad round.
struct RoadLists {
  Front nxt;
  int n_nxt;
  Far far;
  int n_far;
  int *touched;
  int count;
};

// Front entries b .. of one railroad round over nc entries, at most 2P (the wave's batch): the
// neighbours whose distance they improve go to the wave's stage.
template <int P, bool Wide, class Flush>
__device__ __forceinline__ void road_batch(const TraceArgs &a, const Lane<Wide> &ln, const Front &cur, int b, int nc,
                                           unsigned bound, Stage &st, int &staged, Flush &&flush) {
  int u[P];
  const int ue = batch_entries<P>(ln, cur, b, nc, u);
  unsigned long long q = 0, w[P];
  unsigned me = 0;
  if (ln.lane < min(2 * P, nc - b)) {  // lane e: entry e's distance by the dequeue, and its mask
    q = g_or(a.road + ue, kNotQueued);
    me = mask_of(a, ue);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) w[p] = g_ld(word_at(a.road0, ln.at(u[p])));
  const unsigned de = road_dist(q);
  if (de > bound) me = 0;
  staged_pairs<P>([&](int p) {
    const unsigned m = of_entry(ln, me, 2 * p), d = of_entry(ln, de, 2 * p);
    const unsigned lo = unsigned(w[p]), hi = unsigned(w[p] >> 32);
    const float cost = __uint_as_float(lo & kCostBits);
    const bool rail = cost == 0.0f;
    // The step d + cost, on the bits: one ulp up where a positive cost leaves d as it is (the rule of
    // the reference's brook_vw_step, common.cuh:123-127), so distances increase strictly along every
    // step and predecessor walks terminate.
    const unsigned c = rail ? d : max(__float_as_uint(__uint_as_float(d) + cost), d + 1u);
    const bool later = c > bound;  // never a rail: d <= bound
    const unsigned nhi = (c << 1) | unsigned(later);
    const unsigned nlo = (lo & kCostBits) | (rail | later ? unsigned(kNotQueued) : 0u);
    // c below the distance: 2 * distance + far flag is above 2 * c + 1
    stage_put(st, staged, ((m & ln.bit) != 0u) & ((nhi | 1u) < hi), u[p] + ln.off, ((unsigned long long)nhi << 32) | nlo);
  }, flush);
}

// The staged improvements of a wave (full groups, or all of them).
__device__ __forceinline__ void road_minima(const TraceArgs &a, Shared &sh, RoadMins &mins, Stage &st, int &staged, bool all,
                                            const RoadLists &to) {
  stage_take(st, staged, all, [&](bool on, int v, unsigned long long nv) {
    unsigned long long old = 0;  // "nothing changed" unless the atomic says otherwise
    if (on) old = g_min(a.road + v, nv);
    const unsigned ohi = unsigned(old >> 32), cost = road_cost(nv);
    const bool won = old > nv, later = nv & kFarListed, rail = cost == 0u;
    if (won & rail) {
      const unsigned long long key = ((unsigned long long)road_dist(nv) << 32) | unsigned(v);
      mins.rail = key < mins.rail ? key : mins.rail;
    }
    if (won & later) {
      const unsigned long long key = ((unsigned long long)road_dist(nv) << 32) | cost;
      mins.far = key < mins.far ? key : mins.far;
    }
    Appends out;
    if (!out.begin(sh.n, kTouched, ohi == unsigned(kUnreached >> 32), to.n_nxt, won & !later & !rail & (int(unsigned(old)) < 0),
                   to.n_far, won & later & !(ohi & 1u)))
      return;
    // the far lists hold 2 * count entries: a wave whose appends would pass the end writes none
    const int end = out.at[2] + out.count(2);
    const bool full = end > 2 * to.count;
    if (out.set[2] && end > to.count) atomicOr(&sh.flags[to.n_nxt], full ? kLong | kFull : kLong);
    if (ohi == unsigned(kUnreached >> 32)) g_st(to.touched + out.place(0), v);
    if (won & !later & !rail & (int(unsigned(old)) < 0)) to.nxt.put(out.place(1), v);
    if (won & later & !(ohi & 1u) & !full) to.far.put(out.place(2), v);
  });
}

// Far-list compaction between rounds. A voxel can hold several entries: its entry goes stale when
// a near improvement clears its far flag, and it is far-listed anew when a later, smaller bound
// (a closer rail) leaves its next improvement beyond the band. Within one round the bound is fixed,
// so a round appends at most one entry per voxel (at most `count`); a list that holds more than
// `count` entries after a round keeps one entry per far-listed voxel (the one whose atomic clears
// the far flag, restored after a barrier), so 2 * count entries always suffice.
__device__ __forceinline__ void far_compact(const TraceArgs &a, Shared &sh, const Far &from, int n_from, const Far &to,
                                            int n_to) {
  const int nf = sh.n[n_from];
  for (int i = threadIdx.x; i < nf; i += blockDim.x) {
    const int w = from.get(i);
    if (g_and(a.road + w, ~kFarListed) & kFarListed) to.put(wave_slot(&sh.n[n_to]), w);
  }
  __syncthreads();
  const int kept = sh.n[n_to];
  for (int i = threadIdx.x; i < kept; i += blockDim.x) g_or(a.road + to.get(i), kFarListed);
  if (threadIdx.x == 0) sh.n[n_from] = 0;
  __syncthreads();
}

__device__ __forceinline__ float rail_bound(const Shared &sh) {
  float b = sh.T;
  unsigned long long rb = sh.rail_best;
  if (rb != kMaxKey) b = fminf(b, __uint_as_float((unsigned)(rb >> 32)));
  return b;
}

// Returns kRailFound when the nearest rail is settled (sh.rail_best), kNoRail when no rail is
// reachable, kStalled / kOverflowed when the run is given up (see round_budget, far_compact). A
// `source` run never takes t itself for a rail: with no rails in the label it settles every voxel
// reachable from t (the vertex-weighted distances of the fix_branching=False field). The far lists
// hold 2 * count entries.
template <bool Wide>
__device__ __forceinline__ int railroad(const TraceArgs &a, Shared &sh, const Lane<Wide> &ln, int t, int count, const Lists &l,
                                        bool source = false) {
  if (threadIdx.x == 0) {
    g_st(l.touched, t);
    for (int j = 0; j < kCounters; ++j) sh.n[j] = 0;
    for (int j = 0; j < 3; ++j) sh.flags[j] = 0;
    sh.n[kTouched] = 1;
    sh.minfar = kMinfarNone;
    const unsigned cost = road_cost(lp_u64(a.road + t));
    const float ft = __uint_as_float(cost);
    if (ft == 0.0f && !source) {
      sp_u64(a.road + t, road_word(0u, kNotQueued, cost));
      sh.rail_best = (unsigned)t;
      sh.done = kRailFound;
    } else {
      sp_u64(a.road + t, road_word(0u, 0ULL, cost));  // queued
      sh.rail_best = kMaxKey;
      sh.done = 0;
      l.near[0].put(0, t);
      sh.n[0] = 1;
      sh.T = fmaxf(2.0f * ft, 1e-30f);
    }
  }
  __syncthreads();
  RoadMins mins;
  Stage &st = sh.stage[ln.wave];
  Front cur = l.near[0], nxt = l.near[1];
  Far fcur = l.far[0], fnxt = l.far[1];
  int fc = kFar, fn = kFar + 1;  // their lengths are sh.n[fc], sh.n[fn]
  int r = 0;                     // the near list's length is sh.n[r]
  long long rounds = 0;          // rounds and phases so far (the same in every thread)
  const long long budget = round_budget(count);
  auto swap_far = [&] {
    const Far f = fcur; fcur = fnxt; fnxt = f;
    const int n = fc; fc = fn; fn = n;
  };
  int done = sh.done;  // read after a barrier, written again only after the next one
  while (done == 0) {
    int stop = 0;
    for (;;) {  // settle the near band
      const int nc = __builtin_amdgcn_readfirstlane(sh.n[r]);
      if (nc == 0) break;
      const int rn = rot_next(r);
      if (threadIdx.x == 0) {
        sh.n[rot_prev(r)] = sh.flags[rot_prev(r)] = 0;
        sh.prof[5] += 1;
        sh.prof[10] += nc;
      }
      const unsigned bound = unsigned(__builtin_amdgcn_readfirstlane(__float_as_int(rail_bound(sh))));
      const RoadLists to{nxt, rn, fcur, fc, l.touched, count};
      int staged = 0;
      with_pairs<kMaxPairs>(nc, kWaves, [&](auto Pairs) {
        constexpr int P = decltype(Pairs)::value;
        for (int b = ln.wave * 2 * P; b < nc; b += kWaves * 2 * P)
          road_batch<P>(a, ln, cur, b, nc, bound, st, staged, [&] { road_minima(a, sh, mins, st, staged, false, to); });
      });
      road_minima(a, sh, mins, st, staged, true, to);
      road_fold(sh, mins);
      __syncthreads();
      r = rn;
      const Front f = cur; cur = nxt; nxt = f;
      const int flags = sh.flags[r];
      if ((flags & kFull) || ++rounds > budget) { stop = (flags & kFull) ? kOverflowed : kStalled; break; }
      if (flags & kLong) {
        far_compact(a, sh, fcur, fc, fnxt, fn);
        swap_far();
      }
    }
    if (stop) {  // uniform: every thread read the same flags
      done = stop;
      break;
    }
    if (threadIdx.x == 0) {  // phase end: nearest rail final? else advance the band
      unsigned long long rb = sh.rail_best, mf = sh.minfar;
      if (rb != kMaxKey && (__uint_as_float((unsigned)(rb >> 32)) <= sh.T || mf == kMinfarNone)) sh.done = kRailFound;
      else if (mf == kMinfarNone) sh.done = kNoRail;
      else if (rounds + 1 > budget) sh.done = kStalled;
      else {
        float dmin = __uint_as_float((unsigned)(mf >> 32)), f = __uint_as_float((unsigned)mf);
        float w = BROOK_ROAD_BAND * f, lo = 5e-4f * dmin;
        if (!(w > lo)) w = lo;
        sh.T = dmin + w;
        sh.minfar = kMinfarNone;
      }
      sh.prof[8] += 1;
      sh.prof[9] += sh.n[fc];
    }
    ++rounds;
    __syncthreads();
    done = sh.done;
    if (done) break;
    const int nf = sh.n[fc];
    const float bound = rail_bound(sh);
    // Promote far voxels inside the new band. Entries whose far flag is clear are stale (the voxel
    // went near); of several entries of one voxel, the one whose atomic clears the far flag acts.
    // A far-listed word is never queued, so the claim also queues it; a voxel still beyond the
    // band gets both flags back. Each voxel lands in at most one list (at most count entries).
    for (int i = threadIdx.x; i < nf; i += blockDim.x) {
      const int w = fcur.get(i);
      if (!(lp_u64(a.road + w) & kFarListed)) continue;
      const unsigned long long was = g_and(a.road + w, ~(kFarListed | kNotQueued));
      if (!(was & kFarListed)) continue;
      const float dw = __uint_as_float(road_dist(was));
      if (dw <= bound) {
        cur.put(wave_slot(&sh.n[r]), w);
      } else {
        g_or(a.road + w, kFarListed | kNotQueued);
        const unsigned long long key = ((unsigned long long)road_dist(was) << 32) | road_cost(was);
        mins.far = key < mins.far ? key : mins.far;
        fnxt.put(wave_slot(&sh.n[fn]), w);
      }
    }
    road_fold(sh, mins);
    __syncthreads();
    if (threadIdx.x == 0) sh.n[fc] = 0;  // read above; appended to again after the next phase end's barrier
    swap_far();
  }
  return done;
}

// The railroad's words back to unreached, costs kept.
__device__ __forceinline__ void road_restore(const TraceArgs &a, const Shared &sh, const int *touched) {
  const int nt = sh.n[kTouched];
  for (int j = threadIdx.x; j < nt; j += blockDim.x) {
    const int v = g_ld(touched + j);
    sp_u64(a.road + v, kUnreached | road_cost(lp_u64(a.road + v)));
  }
}

// ---- backtrace (wave 0) ---------------------------------------------------------------------
// Lane k probes neighbour k: its word beside the voxel's mask, one memory step per path vertex.
__device__ __forceinline__ void backtrace(const TraceArgs &a, Shared &sh, int t, int count, int *walk) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  const bool on = lane < 26;
  const int off = on ? step_offset(a.d, kNX[lane], kNY[lane], kNZ[lane]) : 0;
  const unsigned rank = on ? unsigned(kD3Rank[on ? lane : 0]) : 64u;
  int cur = (int)(unsigned)(sh.rail_best & 0xFFFFFFFFULL);
  int kept = 0;
  bool first = true;
  for (;;) {
    int kb = -1;
    if (cur != t) {
      const unsigned m = in_mask(a, cur);  // the predecessor's step to cur must be permitted
      const unsigned long long w = lp_u64(a.road + (long long)cur + off);  // padded: readable whatever the mask
      unsigned db = kInfBits;
      if (on && ((m >> lane) & 1u) && road_cost(w) != 0u) db = road_dist(w);
      const unsigned mb = wave_min_u32(db);
      if (mb < kInfBits) kb = __ffsll((long long)ballot(db == mb)) - 1;
    }
    if (first && kb >= 0) {  // the join at u = cur + N[kb]: u's first rail in dijkstra3d order
      const int u = cur + nb_offset(kb, a.d);
      const unsigned mu = mask_of(a, u);
      const unsigned long long w = lp_u64(a.road + (long long)u + off);
      const unsigned r = wave_min_u32(on && ((mu >> lane) & 1u) && road_cost(w) == 0u ? rank : 64u);
      if (r < 26u) {
        int ks = kD3Inv[r];
        cur = u + nb_offset(ks, a.d);
        kb = kOpp[ks];
      }
    }
    first = false;
    if (kept >= count) { kept = -1; break; }  // longer than the label: cannot happen on a valid field
    if (lane == 0) g_st(walk + kept, cur);
    ++kept;
    if (kb < 0) break;
    cur += nb_offset(kb, a.d);
  }
  if (lane == 0) sh.path_len = kept;
}

// ---- fix_branching=False: parent field and parent walk ---------------------------------------
// The field (batched.cu:246-251): the railroad from the root in `source` mode (the near-far
// bands of flood_lab_nf, batched_coop.inc:125-267) gives every voxel of the label its
// vertex-weighted distance over the PDRF; parents_lab (batched_regular.inc:113-134) then takes
// the same-label neighbour of smallest distance, first k on ties (-1 at the root and at voxels the
// run does not reach, as a label that filled holes split has), and the words go back to unreached.
// Returns the railroad's status: kNoRail is the complete field; kRailFound means the run met a
// voxel of PDRF 0 besides the root (it would stop there as at a rail; PDRF underflows to 0 only for
// extreme exponents), and the label is ejected; kStalled / kOverflowed end the label as failed.
template <bool Wide>
__device__ __forceinline__ int parent_field(const TraceArgs &a, Shared &sh, const Lane<Wide> &ln, int root, const int *voxels,
                                            int count, const Lists &l) {
  for (int j = threadIdx.x; j < count; j += blockDim.x) g_st(a.parent + g_ld(voxels + j), -1);  // unreached: no parent
  __syncthreads();
  const int status = railroad(a, sh, ln, root, count, l, true);
  const int nt = sh.n[kTouched];
  constexpr int P = kMaxPairs;
  for (int b = ln.wave * 2 * P; b < nt; b += kWaves * 2 * P) {  // half a wave per voxel, a lane per neighbour
    int v[P];
    unsigned long long w[P];
    unsigned m[P];
#pragma unroll
    for (int p = 0; p < P; ++p) v[p] = g_ld(l.touched + min(b + 2 * p + ln.half, nt - 1));
#pragma unroll
    for (int p = 0; p < P; ++p) {
      m[p] = in_mask(a, v[p]);
      w[p] = g_ld(word_at(a.road0, ln.at(v[p])));
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const unsigned dv = unsigned(__shfl(int(road_dist(w[p])), ln.half * 32 + kCentre, 64));
      const unsigned du = m[p] & ln.bit ? road_dist(w[p]) : kInfBits;
      const unsigned best = half_min(du);
      const unsigned k = half_min(du == best && ln.bit ? unsigned(ln.k) : 64u);  // the first k of equal distances
      const bool has = v[p] != root && dv != 0u && dv < kInfBits && best < kInfBits;
      if (ln.slot == 0) g_st(a.parent + v[p], has ? v[p] + nb_offset(int(k), a.d) : -1);  // (the last voxel repeats past the end)
    }
  }
  __syncthreads();
  road_restore(a, sh, l.touched);
  __syncthreads();
  return status;
}

// The walk (one thread):
// backtrace_parent_lab (lockstep_regular.inc:166-202): from the target along the parent field,
// keeping every vertex up to and including the first without a parent (-1 at the root, STOP -2
// at a vertex an earlier path emitted). The walk is a pointer chase; its length is the path's.
__device__ __forceinline__ void parent_walk(const TraceArgs &a, Shared &sh, int t, int count, int *walk) {
  if (threadIdx.x != 0) return;
  int cur = t, kept = 0;
  for (;;) {
    const int p = lp_i(a.parent + cur);
    if (kept >= count) { kept = -1; break; }  // longer than the label: cannot happen on a valid field
    g_st(walk + kept, cur);
    ++kept;
    if (p < 0) break;
    cur = p;
  }
  sh.path_len = kept;
}

// ---- invalidation ---------------------------------------------------------------------------
// A claim word is (bottleneck bits << 32) | (source + 1) << 1 | queued: claims order by (bottleneck,
// source), and the improving atomic minimum returns whether the voxel is already queued for the next
// round (an equal claim never re-queues). A round's snapshot clears the queued bit with the atomic
// that reads the claim. kFree is unclaimed, kDead invalidated.
//
// An offer whose bottleneck lies beyond the band [.., hi) takes the same atomic minimum: a word at or
// above hi is then a waiting voxel's best offer so far, which no claim of the band depends on. Its
// first offer (old word free) lists the voxel; at the band's end the waiting voxels whose word fell
// into the next band are its first front, already queued. The reference pulls instead: at the band's end
// every waiting voxel takes the smallest (max(bottleneck, distance), source) over its claimed
// neighbours' final claims. Both are the same minimum, because every claimed voxel offers its final
// claim to all its neighbours, with one exception: a voxel whose claim improves after it offered
// (0.2 % of the claims of the 512^3 workload) leaves offers of the old claim behind. Those voxels
// are noted (kStale), and before the band ends their waiting neighbours' words are replaced by
// exact pulls. Measured on that workload's slowest label: 711 k pulls of 26 neighbours each became as
// many single word reads.
__device__ __forceinline__ unsigned claim_low(unsigned su) { return (su + 1u) << 1 | 1u; }
__device__ __forceinline__ unsigned long long claim_word(unsigned mb, unsigned su) {
  return ((unsigned long long)mb << 32) | claim_low(su);
}
__device__ __forceinline__ unsigned claim_source(unsigned long long w) { return ((unsigned)w >> 1) - 1u; }

// The invalidation ball around source s: scale * DBF(s) + constant. Every source of an
// invalidation is a voxel of its path, so the radii are staged once in an LDS table of (source,
// radius) slots, direct-mapped by a multiplicative hash (of colliding path voxels the lowest index
// keeps the slot); a source found in its slot costs no device-memory load, any other is read as
// before. Table and fallback give the same bits (one expression).
__device__ __forceinline__ float ball_radius(const Ball &ball, float dbf) { return ball.scale * dbf + ball.constant; }
__device__ __forceinline__ int radius_slot(unsigned s) { return int((s * 0x9E3779B1u) >> 20); }
static_assert(kRadiusSlots == 1 << 12, "radius_slot yields 12 bits");
__device__ __forceinline__ float source_radius(const TraceArgs &a, const Ball &ball, const unsigned long long *tab,
                                               unsigned s) {
  const unsigned long long e = tab[radius_slot(s)];
  return (unsigned)(e >> 32) == s ? __uint_as_float((unsigned)e) : ball_radius(ball, g_ld(a.dbf + s));
}

// Distance over voxel offsets (whole numbers, exact as floats).
__device__ __forceinline__ float offset_distance(const TraceArgs &a, float ox, float oy, float oz) {
  float dx = a.wx * ox, dy = a.wy * oy, dz = a.wz * oz;
  return sqrtf(dx * dx + dy * dy + dz * dz);
}

// A front entry's snapshot, in the lane that took it.
struct Offer {
  int u = 0;
  unsigned m = 0;                          // neighbours it offers to
  unsigned mu = 0, low = 0;                // its claim's bottleneck; its source as an offer's low half
  float maxd = 0.0f;                       // the source's ball
  float ox = 0.0f, oy = 0.0f, oz = 0.0f;   // its place relative to the source
  __device__ __forceinline__ void set(const TraceArgs &a, const Ball &ball, const Shared &sh, unsigned long long ku) {
    const unsigned su = claim_source(ku);
    mu = unsigned(ku >> 32);
    low = claim_low(su);
    maxd = source_radius(a, ball, sh.radius, su);
    int x, y, z, qx, qy, qz;
    place(a, u, x, y, z);
    place(a, int(su), qx, qy, qz);
    ox = float(x - qx);
    oy = float(y - qy);
    oz = float(z - qz);
  }
};

// Where a round's offers go.
struct OfferLists {
  Front nxt;
  int n_nxt;  // claimed and to be queued
  Far far;
  int n_far;  // waiting
  int *touched, *stale;
  int stale_cap;
  unsigned hi;  // the band's end
};

// Offers of the entries held by lanes from .. from + 2P - 1 (their masks 0 beyond the wave's batch) to
// their neighbours, u the entries and w the neighbours' words, loaded at any time of the round: an
// offer whose bottleneck is above the word's cannot win. The others go to the wave's stage.
template <int P, bool Wide, class Flush>
__device__ __forceinline__ void offer_batch(const TraceArgs &a, const Lane<Wide> &ln, const Offer &e, int from, const int (&u)[P],
                                            const unsigned long long (&w)[P], Stage &st, int &staged, Flush &&flush) {
  staged_pairs<P>([&](int p) {
    const int at = from + 2 * p;
    const unsigned m = of_entry(ln, e.m, at), mu = of_entry(ln, e.mu, at), low = of_entry(ln, e.low, at);
    const float maxd = of_entry(ln, e.maxd, at);
    const float d = offset_distance(a, of_entry(ln, e.ox, at) + ln.dx, of_entry(ln, e.oy, at) + ln.dy, of_entry(ln, e.oz, at) + ln.dz);
    const unsigned mb = max(__float_as_uint(d), mu);  // M = max(M[u], d)
    stage_put(st, staged, ((m & ln.bit) != 0u) & (unsigned(w[p]) != 0u) & (d < maxd) & (unsigned(w[p] >> 32) >= mb),
              u[p] + ln.off, ((unsigned long long)mb << 32) | low);
  }, flush);
}

// The staged offers of a wave (full groups, or all of them). lowest: this thread's least waiting one.
__device__ __forceinline__ void offer_minima(const TraceArgs &a, Shared &sh, Stage &st, int &staged, bool all,
                                             const OfferLists &to, unsigned &lowest) {
  stage_take(st, staged, all, [&](bool on, int v, unsigned long long nv) {
    unsigned long long old = 0;  // "no improvement" unless the atomic says otherwise
    if (on) old = g_min(a.claim + v, nv);
    const unsigned ohi = unsigned(old >> 32), mb = unsigned(nv >> 32);
    const bool won = old > nv, now = mb < to.hi, fresh = ohi >= to.hi;
    const bool claimed = won & now & fresh, waits = won & !now & (ohi == ~0u);
    const bool again = won & now & !fresh & !(unsigned(old) & 1u);  // it had offered its old claim already
    if (won & !now) lowest = min(lowest, mb);
    if (again) {
      const int at = wave_slot(&sh.n[kStale]);
      if (at < to.stale_cap) g_st(to.stale + at, v);
    }
    Appends out;
    if (!out.begin(sh.n, kTouched, claimed, to.n_nxt, claimed | again, to.n_far, waits)) return;
    if (claimed) g_st(to.touched + out.place(0), v);
    if (claimed | again) to.nxt.put(out.place(1), v);
    if (waits) to.far.put(out.place(2), v);
  });
}

// One invalidation round over nc entries: every snapshot before any offer. A wave's entries stay in
// its registers, a lane each, in fronts of up to kHeld per wave (whole batches, so that none reaches past
// lane 63); longer fronts keep their snapshots in device memory. Fronts that fit one batch per wave load
// their neighbours' words before the barrier.
constexpr int kHeld = 64 / (2 * kMaxPairs) * (2 * kMaxPairs);
template <bool Wide>
__device__ __forceinline__ void offer_round(const TraceArgs &a, const Ball &ball, Shared &sh, const Lane<Wide> &ln,
                                            const Front &cur, int nc, const OfferLists &to, unsigned long long *snap,
                                            unsigned &lowest) {
  Stage &st = sh.stage[ln.wave];
  int staged = 0;
  auto flush = [&] { offer_minima(a, sh, st, staged, false, to, lowest); };
  if (nc <= kWaves * 2 * kMaxPairs) {
    with_pairs<kMaxPairs>(nc, kWaves, [&](auto Pairs) {
      constexpr int P = decltype(Pairs)::value;
      const int b = ln.wave * 2 * P;
      Offer e;
      int u[P];
      unsigned long long w[P];
      if (b < nc) {
        e.u = batch_entries<P>(ln, cur, b, nc, u);
        const bool mine = ln.lane < min(2 * P, nc - b);
        unsigned long long ku = 0;
        if (mine) {
          ku = g_and(a.claim + e.u, ~1ULL);
          e.m = mask_of(a, e.u);
        }
#pragma unroll
        for (int p = 0; p < P; ++p) w[p] = g_ld(word_at(a.claim0, ln.at(u[p])));
        if (mine) e.set(a, ball, sh, ku);
      }
      __syncthreads();
      if (b < nc) offer_batch<P>(a, ln, e, 0, u, w, st, staged, flush);
    });
    offer_minima(a, sh, st, staged, true, to, lowest);
    return;
  }
  constexpr int P = kMaxPairs;
  int u[P];
  unsigned long long w[P];
  if (nc <= kWaves * kHeld) {
    const int per = (nc + kWaves - 1) / kWaves, b = ln.wave * per, n = min(per, nc - b);
    Offer e;
    if (ln.lane < n) {
      e.u = cur.get(b + ln.lane);
      e.m = mask_of(a, e.u);
      e.set(a, ball, sh, g_and(a.claim + e.u, ~1ULL));
    }
    __syncthreads();
    for (int from = 0; from < n; from += 2 * P) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        u[p] = int(of_entry(ln, unsigned(e.u), from + 2 * p));
        w[p] = g_ld(word_at(a.claim0, ln.at(u[p])));
      }
      offer_batch<P>(a, ln, e, from, u, w, st, staged, flush);
    }
    offer_minima(a, sh, st, staged, true, to, lowest);
    return;
  }
  for (int i = threadIdx.x; i < nc; i += blockDim.x) g_st(snap + i, g_and(a.claim + cur.get(i), ~1ULL));
  __syncthreads();
  for (int b = ln.wave * 2 * P; b < nc; b += kWaves * 2 * P) {
    Offer e;
    e.u = batch_entries<P>(ln, cur, b, nc, u);
#pragma unroll
    for (int p = 0; p < P; ++p) w[p] = g_ld(word_at(a.claim0, ln.at(u[p])));
    if (ln.lane < min(2 * P, nc - b)) {
      e.m = mask_of(a, e.u);
      e.set(a, ball, sh, g_ld(snap + b + ln.lane));
    }
    offer_batch<P>(a, ln, e, 0, u, w, st, staged, flush);
  }
  offer_minima(a, sh, st, staged, true, to, lowest);
}

// The exact pulls of list entries b .. b + 1 (n of them), a half each: the entry's word, when it waits,
// becomes the smallest (max(bottleneck, distance to the neighbour's source), source) among its
// claimed neighbours whose source's ball holds it, or free. An entry may occur twice: claimed
// words do not change here, so both write the same.
template <bool Wide>
__device__ __forceinline__ void pull_pair(const TraceArgs &a, const Ball &ball, const Shared &sh, const Lane<Wide> &ln, int c,
                                          bool on, unsigned hi) {
  const unsigned m = in_mask(a, c);
  const unsigned long long w = lp_u64(word_at(a.claim0, ln.at(c)));
  unsigned long long best = kMaxKey;
  if ((m & ln.bit) && unsigned(w) != 0u && unsigned(w >> 32) < hi) {
    const unsigned su = claim_source(w);
    int x, y, z, qx, qy, qz;
    place(a, c, x, y, z);
    place(a, int(su), qx, qy, qz);
    const float d = offset_distance(a, float(x - qx), float(y - qy), float(z - qz));
    if (d < source_radius(a, ball, sh.radius, su)) best = claim_word(max(__float_as_uint(d), unsigned(w >> 32)), su);
  }
  best = half_min_u64(best);
  if (on && ln.slot == kCentre && unsigned(w >> 32) >= hi && w != kFree) sp_u64(a.claim + c, best);
}

// The waiting words that stale offers may have set, made exact: those of the noted voxels' neighbours,
// or every waiting one when the notes overflowed. Ends with a barrier.
template <bool Wide>
__device__ __forceinline__ void pull_stale(const TraceArgs &a, const Ball &ball, Shared &sh, const Lane<Wide> &ln, const Far &far,
                                           int nf, int ns, const OfferLists &to, int *dirty) {
  const bool all = ns > to.stale_cap;
  if (!all) {
    for (int i = ln.wave * 2; i < ns; i += kWaves * 2) {
      const int u = g_ld(to.stale + min(i + ln.half, ns - 1));
      const unsigned m = i + ln.half < ns ? mask_of(a, u) : 0u;
      const unsigned long long w = lp_u64(word_at(a.claim0, ln.at(u)));
      if ((m & ln.bit) && unsigned(w >> 32) >= to.hi && w != kFree) {
        const int at = wave_slot(&sh.n[kDirty]);
        if (at < to.stale_cap) g_st(dirty + at, u + ln.off);
      }
    }
    __syncthreads();
  }
  const int nd = sh.n[kDirty];
  const bool listed = !all && nd <= to.stale_cap;
  const int n = listed ? nd : nf;
  for (int i = ln.wave * 2; i < n; i += kWaves * 2) {
    const int j = min(i + ln.half, n - 1);
    pull_pair(a, ball, sh, ln, listed ? g_ld(dirty + j) : far.get(j), i + ln.half < n, to.hi);
  }
  if (threadIdx.x == 0) sh.prof[14] += n;
  __syncthreads();
  if (threadIdx.x == 0) sh.n[kStale] = sh.n[kDirty] = 0;  // appended to again after the promotion's barrier
}

__device__ __forceinline__ int band_of(unsigned mbits, float delta, int kmin) {
  float m = __uint_as_float(mbits);
  int k = (int)(m / delta);
  while ((float)(k + 1) * delta <= m) k++;
  while (k > 0 && (float)k * delta > m) k--;
  return k < kmin ? kmin : k;
}

__device__ __forceinline__ void fold_lowest(unsigned *slot, unsigned &lowest) {
  if (any_lane(lowest != kInfBits)) {
    lowest = wave_min_u32(lowest);
    if (__lane_id() == 0) atomicMin(slot, lowest);
  }
  lowest = kInfBits;
}

// Returns false when the rounds did not converge within the budget (the label is then given up;
// the claimed set still dies).
template <bool Wide>
__device__ __forceinline__ bool invalidate(const TraceArgs &a, const Ball &ball, Shared &sh, const Lane<Wide> &ln,
                                           const int *path, int len, int count, const Lists &l) {
  if (threadIdx.x == 0) {
    for (int j = 0; j < kCounters; ++j) sh.n[j] = 0;
    for (int j = 0; j < 3; ++j) sh.lowest[j] = kInfBits;
  }
  for (int j = threadIdx.x; j < kRadiusSlots; j += blockDim.x) sh.radius[j] = kMaxKey;
  __syncthreads();
  OfferLists to{l.near[1], 1, l.far[0], kFar, l.touched, l.stale, 2 * count, 0u};
  Front cur = l.near[0];
  Far keep = l.far[1];
  int r = 0;   // the current front's length is sh.n[r]
  int bt = 0;  // bands so far mod 3: the waiting list's length is sh.n[kFar + bt], its minimum sh.lowest[bt]
  for (int j = threadIdx.x; j < len; j += blockDim.x) {  // sources: path voxels still alive
    int p = g_ld(path + j);
    atomicMin(&sh.radius[radius_slot(unsigned(p))],
              ((unsigned long long)unsigned(p) << 32) | __float_as_uint(ball_radius(ball, g_ld(a.dbf + p))));
    if (g_cas(a.claim + p, kFree, claim_word(0u, unsigned(p))) == kFree) {
      cur.put(wave_slot(&sh.n[0]), p);
      g_st(l.touched + wave_slot(&sh.n[kTouched]), p);
    }
  }
  __syncthreads();
  long long rounds = 0;  // rounds and bands so far (the same in every thread)
  const long long budget = round_budget(count);
  bool converged = true;
  int band = 0;  // the same in every thread
  unsigned lowest = kInfBits;
  for (;;) {
    to.hi = unsigned(__builtin_amdgcn_readfirstlane(__float_as_int((float)(band + 1) * a.delta)));
    to.n_far = kFar + bt;
    for (;;) {  // synchronous rounds inside the band
      const int nc = __builtin_amdgcn_readfirstlane(sh.n[r]);
      if (nc == 0) break;
      if (++rounds > budget) { converged = false; break; }
      to.n_nxt = rot_next(r);
      if (threadIdx.x == 0) { sh.n[rot_prev(r)] = 0; sh.prof[6] += 1; sh.prof[11] += nc; }
      offer_round(a, ball, sh, ln, cur, nc, to, l.snap, lowest);
      fold_lowest(&sh.lowest[bt], lowest);
      __syncthreads();
      r = to.n_nxt;
      const Front f = cur; cur = to.nxt; to.nxt = f;
    }
    const int nf = sh.n[kFar + bt];
    if (nf == 0 || !converged || ++rounds > budget) { converged = converged && nf == 0; break; }
    if (threadIdx.x == 0) { sh.prof[12] += nf; sh.prof[13] += 1; }
    const int ns = sh.n[kStale];
    // The promotion below appends to the counter that every wave left the rounds by reading as 0: none
    // may append before all have read it (a wave that read an append would begin a round of its own).
    __syncthreads();
    if (ns) pull_stale(a, ball, sh, ln, to.far, nf, ns, to, reinterpret_cast<int *>(l.snap));
    // The next band: the one that holds the least waiting offer (an offer replaced since leaves it
    // too low at worst: an empty band).
    const unsigned least = sh.lowest[bt];
    if (least != kInfBits) band = band_of(least, a.delta, band + 1);
    const unsigned next_hi = __float_as_uint((float)(band + 1) * a.delta);
    const int bn = rot_next(bt);
    for (int i = threadIdx.x; i < nf; i += blockDim.x) {  // promote / keep waiting / drop
      const int c = to.far.get(i);
      const unsigned long long w = lp_u64(a.claim + c);
      const unsigned mb = unsigned(w >> 32);
      if (mb < to.hi || w == kFree) continue;  // claimed in the band; its offer was stale
      if (mb < next_hi) {                      // its word is the claim, queued
        g_st(l.touched + wave_slot(&sh.n[kTouched]), c);
        cur.put(wave_slot(&sh.n[r]), c);
      } else {
        keep.put(wave_slot(&sh.n[kFar + bn]), c);
        lowest = min(lowest, mb);
      }
    }
    fold_lowest(&sh.lowest[bn], lowest);
    if (threadIdx.x == 0) {  // the third slots: last read a band ago, next written a band on
      sh.n[kFar + rot_next(bn)] = 0;
      sh.lowest[rot_next(bn)] = kInfBits;
    }
    __syncthreads();
    const Far f = to.far; to.far = keep; keep = f;
    bt = bn;
  }
  __syncthreads();
  const int nt = sh.n[kTouched];
  if (threadIdx.x == 0) {
    g_add(reinterpret_cast<unsigned long long *>(a.counters + 6), (unsigned long long)nt);
    if (!converged) report_failure(a, kStalled);
  }
  for (int j = threadIdx.x; j < nt; j += blockDim.x) sp_u64(a.claim + g_ld(l.touched + j), kDead);  // the claimed set dies
  __syncthreads();
  return converged;
}

// ---- target selection -----------------------------------------------------------------------
__device__ __forceinline__ int next_target(const TraceArgs &a, Shared &sh, int L) {
  if (threadIdx.x == 0) {
    int pc = sh.pcount;
    sh.ordered = 0;
    if (pc >= g_ld(a.maxp + L)) sh.target = -1;
    else if (pc < g_ld(a.mcount + L)) sh.target = g_ld(a.mflat + g_ld(a.mstart + L) + pc);
    else sh.target = -2;
  }
  __syncthreads();
  if (sh.target != -2) return sh.target;
  const int per = 4, window = per * blockDim.x;
  for (;;) {
    long long c = sh.cursor, e = sh.seg_end;
    if (c >= e) {  // the order is spent: the extra targets after it, last given first (trace.cu:197-199)
      __syncthreads();
      if (threadIdx.x == 0) {
        const int after = a.acount ? g_ld(a.acount + L) : 0;
        if (sh.after_used < after) {
          sh.target = g_ld(a.mflat + g_ld(a.mstart + L) + g_ld(a.mcount + L) + sh.after_used);
          sh.after_used += 1;
        } else {
          sh.target = -1;
        }
      }
      __syncthreads();
      return sh.target;
    }
    if (threadIdx.x == 0) sh.found = INT32_MAX;
    __syncthreads();
    for (int r = 0; r < per; ++r) {
      long long j = c + r * blockDim.x + threadIdx.x;
      if (j < e) {
        int v = g_ld(a.order + j);
        if (lp_u64(a.claim + v) != kDead) atomicMin(&sh.found, int(j - c));
      }
    }
    __syncthreads();
    if (sh.found != INT32_MAX) {
      __syncthreads();
      if (threadIdx.x == 0) {
        sh.cursor = c + sh.found;
        sh.target = g_ld(a.order + c + sh.found);
        sh.ordered = 1;
      }
      __syncthreads();
      return sh.target;
    }
    __syncthreads();
    if (threadIdx.x == 0) sh.cursor = c + window;
    __syncthreads();
  }
}

// ---- somata ------------------------------------------------------------------------------------
// Physical distance from the soma root above the soma radius, in float64 as numpy's
// norm(anisotropy_f32 * (vertex - root)) (lockstep_regular.inc:35-45).
__device__ __forceinline__ bool soma_far(const TraceArgs &a, int v, int rx, int ry, int rz, double radius) {
  int x, y, z;
  unravel(v, a.d, x, y, z);
  const double dx = (double)a.wx * ((double)x - (double)rx), dy = (double)a.wy * ((double)y - (double)ry),
               dz = (double)a.wz * ((double)z - (double)rz);
  double ss = dx * dx + dy * dy;
  ss = ss + dz * dz;
  return sqrt(ss) > radius;
}

// One thread: a soma's walk compacted in place to the vertices Kimimaro keeps
// (lockstep_regular.inc:128-147, 184-195). A railroad walk runs rail end -> target: the target
// and the far vertices stay, and a rail end within the radius is replaced by the root. A parent
// walk runs target -> root: the far vertices and the root stay. Every write lands at or before
// the entry just read, except that a walk of one vertex gets two entries (a label has more voxels).
__device__ __forceinline__ void soma_trim(const TraceArgs &a, Shared &sh, int *walk, int root, double radius) {
  int rx, ry, rz;
  unravel(root, a.d, rx, ry, rz);
  const int n = sh.path_len;
  int kept = 0;
  for (int j = 0; j < n; ++j) {
    const int v = g_ld(walk + j);
    const bool far = soma_far(a, v, rx, ry, rz, radius);
    if (!a.parent && j == 0 && !far) g_st(walk + kept++, root);
    if (far || j == n - 1) g_st(walk + kept++, v);
  }
  sh.path_len = kept;
}

// The somata's own balls (lockstep.cu:197-206), one workgroup per soma label, before the trace:
// the ball of the soma parameters around the root dies, and the label's path budget becomes its
// voxel count minus what the ball took (or max_paths), none when the manual targets reach it.
template <bool Wide>
__global__ void __launch_bounds__(kBlock) soma_balls(const TraceArgs *__restrict__ all, const int2 *__restrict__ queue,
                                                    int nqueue) {
  __shared__ Shared sh;
  const int2 q = queue[blockIdx.x];
  const TraceArgs a = all[__builtin_amdgcn_readfirstlane(q.x)];
  const int L = __builtin_amdgcn_readfirstlane(q.y);
  const Lane<Wide> ln = lane_of<Wide>(a.d);
  const int seg = __builtin_amdgcn_readfirstlane(g_ld(a.seg_start + L));  // uniform: scalar registers
    const int count = __builtin_amdgcn_readfirstlane(g_ld(a.seg_count + L));
  const Lists l = lists_of(a, sh, seg);
  const SomaLabel *soma = a.soma + L;
  if (threadIdx.x == 0) {
    for (int j = 0; j < kProf; ++j) sh.prof[j] = 0;
    g_st(l.walk, int(g_ld(a.root + L)));
  }
  __syncthreads();
  invalidate(a, soma->ball, sh, ln, l.walk, 1, count, l);
  if (threadIdx.x == 0) {
    const long long limit = g_ld(&soma->max_paths);
    const long long budget = limit >= 0 ? limit : (long long)count - sh.n[kTouched];
    const int manual = g_ld(a.mcount + L) + (a.acount ? g_ld(a.acount + L) : 0);
    g_st(a.maxp + L, manual >= budget ? 0 : int(budget < INT32_MAX ? budget : INT32_MAX));
  }
}

// The queue is sorted largest first. Workgroup w < nfixed (the workgroups resident from the start,
// at most the queue's length) takes item w first; every other item comes from the shared cursor,
// from item nfixed on. Workgroups go to the XCDs in turn (w mod 8), so the largest labels start on
// different XCDs instead of wherever the first atomics land, and no XCD's L2 carries more than
// its share of them.
template <bool Wide>
__global__ void __launch_bounds__(kBlock) trace_labels(const TraceArgs *__restrict__ all, const int2 *__restrict__ queue,
                                                      int nqueue, int nfixed, int *next) {
  __shared__ Shared sh;
  __shared__ int item;
  for (bool first_item = true;; first_item = false) {
    __syncthreads();
    if (threadIdx.x == 0) item = first_item && int(blockIdx.x) < nfixed ? int(blockIdx.x) : nfixed + g_add(next, 1);
    __syncthreads();
    if (item >= nqueue) return;
    const int2 q = queue[item];
    const int sample = __builtin_amdgcn_readfirstlane(q.x);
    const TraceArgs a = all[sample];  // uniform: scalar registers
    const int L = __builtin_amdgcn_readfirstlane(q.y);
    const Lane<Wide> ln = lane_of<Wide>(a.d);
    const int seg = __builtin_amdgcn_readfirstlane(g_ld(a.seg_start + L));  // uniform: scalar registers
    const int count = __builtin_amdgcn_readfirstlane(g_ld(a.seg_count + L));
    const Lists l = lists_of(a, sh, seg);
    int *walk = l.walk;
    if (threadIdx.x == 0) {
      sh.cursor = seg;
      sh.seg_end = (long long)seg + count;
      sh.pcount = 0;
      sh.after_used = 0;
      for (int j = 0; j < kProf; ++j) sh.prof[j] = 0;
      sh.tick = wall_clock64();
    }
    const long long label_begin = wall_clock64();
    __syncthreads();
    bool traceable = true;
    if (a.parent) {
      const int field = parent_field(a, sh, ln, int(g_ld(a.root + L)), a.order + seg, count, l);
      lap(sh, 2);
      traceable = field == kNoRail;
      if (field == kRailFound && threadIdx.x == 0) g_st(a.ejected + g_add(a.counters + 2, 1) % a.ejected_cap, L);
      if ((field == kStalled || field == kOverflowed) && threadIdx.x == 0) report_failure(a, field);
    }
    // A soma's paths keep only the vertices beyond its radius (its ball died in soma_balls).
    const bool soma = a.soma && g_ld(&a.soma[L].radius) >= 0.0;
    for (; traceable;) {
      const int t = next_target(a, sh, L);
      lap(sh, 1);
      if (t < 0) break;
      int status = kRailFound;
      if (a.parent) {
        parent_walk(a, sh, t, count, walk);
        if (threadIdx.x == 0) sh.n[kTouched] = 0;
      } else {
        status = railroad(a, sh, ln, t, count, l);
        lap(sh, 2);
        if (status == kRailFound) backtrace(a, sh, t, count, walk);
      }
      __syncthreads();
      lap(sh, 3);
      const int nt = sh.n[kTouched];
      road_restore(a, sh, l.touched);
      if (status == kStalled || status == kOverflowed) {  // given up: the host raises
        if (threadIdx.x == 0) report_failure(a, status);
        __syncthreads();
        break;
      }
      if (status == kNoRail) {
        // No rail reachable from t (a component that filled holes split): as the reference's
        // per-component tracer does for such a label (trace.cu:198-215), an ordered target ends
        // the label with the paths it has, a manual one counts as an empty path.
        if (sh.ordered) break;
        if (threadIdx.x == 0) sh.path_len = 0;
        __syncthreads();
      } else if (sh.path_len < 0) {
        if (threadIdx.x == 0) g_st(a.ejected + g_add(a.counters + 2, 1) % a.ejected_cap, L);
        __syncthreads();
        break;
      }
      if (soma && threadIdx.x == 0) soma_trim(a, sh, walk, int(g_ld(a.root + L)), g_ld(&a.soma[L].radius));
      __syncthreads();
      const int len = sh.path_len;
      if (threadIdx.x == 0 && len > 0) {
        g_add(reinterpret_cast<unsigned long long *>(a.counters + 4), (unsigned long long)nt);
        int pos = g_add(a.counters + 0, len);
        int rec = g_add(a.counters + 1, 1);
        if ((long long)pos + len > a.store_cap || rec >= a.rec_cap) {
          g_or(a.counters + 3, 1);  // overflow: reported to the host
          sh.store_pos = -1;
        } else {
          sh.store_pos = pos;
          g_st(a.rec_label + rec, L);
          g_st(a.rec_len + rec, len);
          g_st(a.rec_start + rec, pos);
        }
      }
      __syncthreads();
      const int pos = sh.store_pos;
      for (int j = threadIdx.x; j < len; j += blockDim.x) {
        int v = g_ld(walk + j);
        if (pos >= 0) g_st(a.store + pos + (len - 1 - j), v);
        if (a.parent) {
          if (!soma) g_st(a.parent + v, -2);  // STOP: later walks end on this vertex (not for somata)
        }
        else sp_u64(a.road + v, kUnreached);    // the path becomes rail (cost 0)
      }
      __syncthreads();
      const bool converged = invalidate(a, a.ball, sh, ln, walk, len, count, l);
      lap(sh, 4);
      if (!converged) break;  // reported by invalidate; the host raises
      if (threadIdx.x == 0) { sh.pcount += 1; sh.prof[7] += 1; }
      __syncthreads();
    }
    if (threadIdx.x == 0 && a.label_stats) {
      sh.prof[0] = (unsigned long long)(wall_clock64() - label_begin);
      for (int j = 0; j < kProf; ++j) g_st(a.label_stats + (long long)kProf * L + j, sh.prof[j]);
    }
  }
}

}  // namespace

void trace_all(Context &ctx, const std::vector<TraceArgs> &args, const std::vector<LabelItem> &items,
               const std::vector<LabelItem> &somata) {
  if (items.empty()) return;
  Buffer<TraceArgs> args_dev(ctx, args.size());
  args_dev.upload(ctx, args.data(), args.size());
  std::vector<int2> q(items.size());
  for (size_t i = 0; i < items.size(); ++i) q[i] = make_int2(items[i].sample, items[i].label);
  Buffer<int2> queue(ctx, q.size());
  queue.upload(ctx, q.data(), q.size());
  Buffer<int> next(ctx, 1);  // queue cursor
  next.clear(ctx);
  const int nq = int(q.size());
  bool wide = false;  // one launch serves every sample of the group
  for (const TraceArgs &t : args) wide |= !narrow_words(t.d);
  // every workgroup takes labels from the queue until it is spent, so any grid drains it
  const int grid = std::min(nq, BROOK_TRACE_GRID > 0 ? BROOK_TRACE_GRID : ctx.compute_units() * 2);
  if (!somata.empty()) {
    std::vector<int2> sq(somata.size());
    for (size_t i = 0; i < somata.size(); ++i) sq[i] = make_int2(somata[i].sample, somata[i].label);
    Buffer<int2> soma_queue(ctx, sq.size());
    soma_queue.upload(ctx, sq.data(), sq.size());
    KernelTimer kt(ctx, "soma_balls");
    (wide ? soma_balls<true> : soma_balls<false>)<<<unsigned(sq.size()), kBlock, 0, ctx.stream()>>>(args_dev.data(), soma_queue.data(), int(sq.size()));
    BROOK_LAUNCHED();
  }
  {
    KernelTimer kt(ctx, "trace_labels");
    (wide ? trace_labels<true> : trace_labels<false>)<<<grid, kBlock, 0, ctx.stream()>>>(args_dev.data(), queue.data(), nq,
                                                    std::min(grid, ctx.compute_units()), next.data());
    BROOK_LAUNCHED();
  }
}

}  // namespace brook
