// The label workgroups' kernels (prepare_labels, soma_balls, trace_labels) on the CPU, one workgroup
// over one label at a time, under schedules that run waves far apart between barriers: every schedule has
// to reach the same barriers and give the same fields, paths and claims. Prints a digest per case; a build
// with one wave per workgroup, where no wave can be ahead of another, prints the digests to be met.
// flood_device.inc and trace_device.inc are the device parts of fields.hip and trace.hip.
#include <hip/hip_runtime.h>

#include "common.hpp"
#define wave_slot(counter) emu::slot(counter)
#include "fields.hpp"
#include "front.hpp"
#include "trace.hpp"
#include "tuned.hpp"
namespace flood_part {
#include "flood_device.inc"
}
namespace trace_part {
#include "trace_device.inc"
}

using namespace brook;
using u64 = unsigned long long;

namespace {

struct Case {
  const char *name;
  Dims d;
  int kind;        // 0: random blob, 1: straight tube, 2: sheet
  bool parents, wide, soma, graph;
  float scale, constant;
};

struct Input {
  Case c;
  std::vector<unsigned> mask, inmask;
  std::vector<float> pdrf, dbf;
  std::vector<int> vox, order;
  std::vector<u64> words;  // padded
  long long pad;
};

Input make(const Case &c, unsigned seed) {
  std::mt19937 rng(seed);
  auto unit = [&] { return float(rng() >> 8) / float(1 << 24); };
  const Dims d = c.d;
  const int n = d.sx * d.sy * d.sz;
  std::vector<char> in(size_t(n), 0);
  for (int v = 0; v < n; ++v) in[size_t(v)] = c.kind == 0 ? unit() < 0.6f : 1;
  Input q{c, std::vector<unsigned>(size_t(n), 0u), {}, std::vector<float>(size_t(n)), std::vector<float>(size_t(n)), {}, {}, {}, word_pad(d)};
  for (int v = 0; v < n; ++v) {
    if (!in[size_t(v)]) continue;
    const int x = v % d.sx, y = v / d.sx % d.sy, z = v / d.sx / d.sy;
    for (int k = 0; k < 26; ++k) {
      const int a = x + kDX[k], b = y + kDY[k], e = z + kDZ[k];
      if (a < 0 || b < 0 || e < 0 || a >= d.sx || b >= d.sy || e >= d.sz) continue;
      if (in[size_t(a + d.sx * (b + d.sy * e))]) q.mask[size_t(v)] |= 1u << k;
    }
  }
  std::vector<int> stack;  // one component, of the first voxel with a neighbour
  std::vector<char> seen(size_t(n), 0);
  for (int v = 0; v < n && stack.empty(); ++v)
    if (q.mask[size_t(v)]) stack.push_back(v), seen[size_t(v)] = 1;
  while (!stack.empty()) {
    const int v = stack.back();
    stack.pop_back();
    for (int k = 0; k < 26; ++k)
      if (q.mask[size_t(v)] >> k & 1u) {
        const int u = v + kDX[k] + d.sx * (kDY[k] + d.sy * kDZ[k]);
        if (!seen[size_t(u)]) seen[size_t(u)] = 1, stack.push_back(u);
      }
  }
  q.words.assign(size_t(n + 2 * q.pad), 0x5555555555555555ULL);  // pads and background: whatever is there
  for (int v = 0; v < n; ++v) {
    if (!seen[size_t(v)]) { q.mask[size_t(v)] = 0; continue; }
    q.vox.push_back(v);
    q.pdrf[size_t(v)] = 0.5f + 8.0f * unit() * unit();
    q.dbf[size_t(v)] = 0.5f + 2.5f * unit();
  }
  if (c.graph) {  // some steps not permitted; pulls are the permitted pushes from the other end
    q.inmask.assign(size_t(n), 0u);
    for (int v : q.vox)
      for (int k = 0; k < 26; ++k)
        if (unit() < 0.1f) q.mask[size_t(v)] &= ~(1u << k);
    for (int v : q.vox)
      for (int k = 0; k < 26; ++k)
        if (q.mask[size_t(v)] >> k & 1u) q.inmask[size_t(v + kDX[k] + d.sx * (kDY[k] + d.sy * kDZ[k]))] |= 1u << kOpp[k];
  }
  q.order = q.vox;
  for (size_t i = q.order.size(); i > 1; --i) std::swap(q.order[i - 1], q.order[rng() % i]);
  if (c.kind == 1) std::reverse(q.order.begin(), q.order.end()), std::sort(q.order.begin(), q.order.end(), std::greater<int>());
  return q;
}

u64 digest(u64 h, const void *p, size_t bytes) {
  const unsigned char *b = static_cast<const unsigned char *>(p);
  for (size_t i = 0; i < bytes; ++i) h = (h ^ b[i]) * 1099511628211ULL;
  return h;
}

struct Lists {
  std::vector<int> l[6];
  std::vector<u64> snap[2];
  explicit Lists(size_t count) {
    for (int i = 0; i < 6; ++i) l[i].resize(count * (i == 2 || i == 3 ? 2 : 1));
    for (auto &s : snap) s.resize(count);
  }
};

u64 flood(const Input &q, const emu::Schedule &schedule, float free_radius) {
  using namespace flood_part::brook;
  const size_t n = q.mask.size(), count = q.vox.size();
  std::vector<u64> road(q.words);
  for (int v : q.vox) road[size_t(v + q.pad)] = kFloodFree;
  Lists lists(count);
  std::vector<float> daf(n, -1.0f), W(26);
  for (int k = 0; k < 26; ++k) W[size_t(k)] = std::sqrt(float(kDX[k] * kDX[k] + kDY[k] * kDY[k] + 4 * kDZ[k] * kDZ[k]));
  const int start[2] = {0, 0}, counts[2] = {0, int(count)};
  const long long first[2] = {-1, q.vox[0]};
  long long root[2] = {-1, -1}, target[2] = {-1, -1};
  float max_daf[2] = {0, 0};
  const float radius[2] = {0, free_radius};
  FloodJob j;
  j.d = q.c.d;
  j.t.seg_start = start;
  j.t.seg_count = counts;
  j.t.vox = q.vox.data();
  j.t.first = first;
  j.t.root = root;
  j.t.target = target;
  j.t.max_daf = max_daf;
  j.t.weights = W.data();
  j.t.free_radius = radius;
  j.t.mask = q.mask.data();
  j.t.road0 = road.data();
  j.t.road = road.data() + q.pad;
  j.daf = daf.data();
  j.lists_a = lists.l[0].data();
  j.lists_b = lists.l[1].data();
  j.far_a = lists.l[2].data();
  j.far_b = lists.l[3].data();
  const int2 queue[1] = {make_int2(0, 1)};
  int next = 0, stalled = 0;
  emu::run(kFloodBlock, schedule, [&] {
    if (q.c.wide) prepare_labels<true>(&j, queue, 1, 1, &next, &stalled);
    else prepare_labels<false>(&j, queue, 1, 1, &next, &stalled);
  });
  u64 h = 14695981039346656037ULL;
  h = digest(h, daf.data(), n * 4);
  h = digest(h, road.data(), road.size() * 8);
  h = digest(h, root, sizeof(root));
  h = digest(h, target, sizeof(target));
  h = digest(h, max_daf, sizeof(max_daf));
  h = digest(h, &stalled, 4);
  return h;
}

u64 trace(const Input &q, const emu::Schedule &schedule, u64 *stats) {
  using namespace trace_part::brook;
  const size_t n = q.mask.size(), count = q.vox.size();
  std::vector<u64> road(q.words), claim(q.words);
  for (int v : q.vox) {
    road[size_t(v + q.pad)] = kUnreached | __float_as_uint(q.pdrf[size_t(v)]);
    claim[size_t(v + q.pad)] = kFree;
  }
  const long long root[2] = {-1, q.vox[0]};
  if (!q.c.parents) road[size_t(root[1] + q.pad)] = kUnreached;
  Lists lists(count);
  const int start[2] = {0, 0}, counts[2] = {0, int(count)}, mstart[2] = {0, 0}, mcount[2] = {0, 1}, acount[2] = {0, 1};
  const int mflat[2] = {q.order[0], q.vox.back()};
  int maxp[2] = {0, INT32_MAX}, counters[16] = {}, ejected[4] = {};
  std::vector<int> store(3 * count + 64), rec_label(count + 8), rec_len(count + 8), rec_start(count + 8), parent(n, -1);
  std::vector<u64> label_stats(2 * kTraceProfileSlots);
  SomaLabel soma[2];
  soma[1].radius = 3.0;
  soma[1].ball = Ball{0.5f, 2.0f};
  TraceArgs a;
  a.d = q.c.d;
  a.by_row = fast_div(unsigned(a.d.sx));
  a.by_plane = fast_div(unsigned(a.d.sx) * unsigned(a.d.sy));
  a.mask = q.mask.data();
  a.road0 = road.data();
  a.road = road.data() + q.pad;
  a.claim0 = claim.data();
  a.claim = claim.data() + q.pad;
  a.dbf = q.dbf.data();
  a.seg_start = start;
  a.seg_count = counts;
  a.order = q.order.data();
  a.mstart = mstart;
  a.mcount = mcount;
  a.mflat = mflat;
  a.acount = acount;
  a.maxp = maxp;
  for (int i = 0; i < 6; ++i) a.lists[i] = lists.l[i].data();
  for (int i = 0; i < 2; ++i) a.snaps[i] = lists.snap[i].data();
  a.store = store.data();
  a.store_cap = (long long)store.size();
  a.rec_label = rec_label.data();
  a.rec_len = rec_len.data();
  a.rec_start = rec_start.data();
  a.rec_cap = int(rec_len.size());
  a.counters = counters;
  a.label_stats = label_stats.data();
  a.ejected = ejected;
  a.ejected_cap = 4;
  a.wz = 2;
  a.ball = Ball{q.c.scale, q.c.constant};
  a.parent = q.c.parents ? parent.data() : nullptr;
  a.root = root;
  a.soma = q.c.soma ? soma : nullptr;
  a.inmask = q.c.graph ? q.inmask.data() : nullptr;
  const int2 queue[1] = {make_int2(0, 1)};
  int next = 0;
  if (q.c.soma)
    emu::run(kBlock, schedule, [&] {
      if (q.c.wide) soma_balls<true>(&a, queue, 1);
      else soma_balls<false>(&a, queue, 1);
    });
  emu::run(kBlock, schedule, [&] {
    if (q.c.wide) trace_labels<true>(&a, queue, 1, 1, &next);
    else trace_labels<false>(&a, queue, 1, 1, &next);
  });
  for (int i = 0; i < kTraceProfileSlots; ++i) stats[i] += label_stats[size_t(kTraceProfileSlots + i)];
  if (counters[2] || counters[3] || counters[8]) std::printf("%s: ejected %d, overflow %d, failed %d\n", q.c.name, counters[2], counters[3], counters[8]);
  u64 h = 14695981039346656037ULL;
  h = digest(h, counters, 8);
  h = digest(h, counters + 6, 8);
  h = digest(h, store.data(), store.size() * 4);
  h = digest(h, rec_len.data(), rec_len.size() * 4);
  h = digest(h, claim.data(), claim.size() * 8);
  h = digest(h, road.data(), road.size() * 8);
  return digest(h, maxp, sizeof(maxp));
}

}  // namespace

int main() {
  const Case cases[] = {{"blob", {24, 17, 9}, 0, false, false, false, false, 1.0f, 1.0f},
                        {"wide words", {13, 9, 21}, 0, false, true, false, false, 1.5f, 0.5f},
                        {"parents", {19, 16, 8}, 0, true, false, false, false, 1.0f, 1.0f},
                        {"soma", {17, 15, 11}, 0, false, false, true, false, 1.0f, 1.5f},
                        {"graph", {21, 18, 7}, 0, false, false, false, true, 1.2f, 1.0f},
                        {"tube", {250, 2, 2}, 1, false, false, false, false, 0.5f, 1.0f},
                        {"sheet", {47, 41, 1}, 2, false, false, false, false, 2.0f, 3.0f},
                        {"sheet on edge", {29, 1, 33}, 0, false, false, false, false, 1.0f, 2.0f},
                        {"column", {1, 1, 90}, 2, true, false, false, false, 1.0f, 1.0f}};
  const int waves = trace_part::brook::kWaves;
  std::vector<emu::Schedule> schedules;
  for (int s = 0; s < std::min(waves, 2); ++s) {  // the first or the last wave ahead of the others
    emu::Schedule o;
    for (int w = 0; w < waves; ++w) o.order.push_back(s ? waves - 1 - w : w);
    schedules.push_back(o);
  }
  for (unsigned seed = 1; waves > 1 && seed <= 2; ++seed) schedules.push_back(emu::Schedule{{}, seed});
  u64 stats[kTraceProfileSlots] = {};
  for (const Case &c : cases) {
    const Input q = make(c, 7u);
    u64 want[3] = {};
    for (size_t s = 0; s < schedules.size(); ++s) {
      const u64 got[3] = {flood(q, schedules[s], 0.0f), flood(q, schedules[s], 3.0f), trace(q, schedules[s], stats)};
      for (int i = 0; i < 3; ++i) {
        if (s == 0) want[i] = got[i];
        if (got[i] != want[i]) {
          std::printf("%s: schedule %zu gives other %s\n", c.name, s, i == 2 ? "paths" : "fields");
          return 1;
        }
      }
    }
    std::printf("%s %016llx %016llx %016llx\n", c.name, want[0], want[1], want[2]);
    std::fflush(stdout);
  }
  std::fprintf(stderr, "railroad rounds %llu, invalidation rounds %llu, paths %llu, waiting %llu, bands %llu, pulled %llu\n", stats[5],
               stats[6], stats[7], stats[12], stats[13], stats[14]);
  return 0;
}
