// Canonical postprocess of packed skeletons on the device (post.cu:1-651, post_kernels.cuh:1-407:
// Kimimaro 5.8.1's remove_dust, remove_loops, join_close_components and remove_ticks with the
// reference's tie rules).
//
// Whole-result passes are wide: union-find components over every edge, per-edge lengths, keep
// masks and prefix sums, radix sorts of edge keys and of join candidates, a 27-cell grid search
// for join candidates. The rules that are sequential by nature (one component's cycle loop, one
// tree's tick loop, one label's greedy fusion) are chains of dependent accesses: rows, neighbour lists
// (doubly linked in insertion order, with a free list), search stack and path for the loops; a CSR
// neighbour table, chain records, end slots and a binary heap keyed (length, lower end, higher end) for
// the ticks. A component (a tree) is one wave's: all lanes take the same steps on the same
// addresses, so no step diverges, scans over its vertices, rows or cycle use all of them, and its
// state, in 16-bit indices, lies in LDS up to kLdsPiece bytes (about 2700 vertices) and in device
// memory beyond. One lane per component of a 64-lane wave, state in device memory, took 11.5 ms for
// the loops and 5.1 ms for the ticks of 150 skeletons of 1100 vertices each; a wave each with its
// state in LDS takes 1.7 and 0.7 ms.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <stdexcept>

#include "common.hpp"
#include "post.hpp"

#pragma clang fp contract(off)

namespace brook {
namespace {

constexpr int kThreads = 256;
constexpr unsigned long long kNone = ~0ULL;
unsigned grid(long long n) { return unsigned(std::max<long long>(1, (n + kThreads - 1) / kThreads)); }

template <class Op> void with_scratch(Context &ctx, Buffer<unsigned char> &scratch, Op &&op) {
  size_t bytes = 0;
  BROOK_HIP(op(nullptr, bytes));
  if (bytes > scratch.size()) scratch = Buffer<unsigned char>(ctx, std::max<size_t>(bytes, 1));
  BROOK_HIP(op(scratch.data(), bytes));
}

// Bits of the keys 0 .. n.
int bits_for(long long n) {
  int bits = 1;
  while ((1LL << bits) <= n) ++bits;
  return bits;
}

template <class T> T read_one(Context &ctx, const T *p) {
  T v{};
  BROOK_HIP(hipMemcpyAsync(&v, p, sizeof(T), hipMemcpyDeviceToHost, ctx.stream()));
  ctx.synchronize();
  return v;
}

// ---------------------------------------------------------------------------------------------
// one wave per component: LDS address space, wave-wide steps

template <class T> using InLds = __attribute__((address_space(3))) T;
template <class T> using InGlobal = __attribute__((address_space(1))) T;
constexpr size_t kLdsPiece = 150 * 1024;

// Lanes see what other lanes of the wave wrote (blocks of one wave).
__device__ __forceinline__ void wave_sync() { __syncthreads(); }

// The greater (Sign 1) or smaller (Sign -1) value over the lanes that have one (index >= 0), the
// lower index on ties; every lane gets the index, -1 if none has.
template <int Sign> __device__ __forceinline__ int wave_extreme(float d, int index) {
  for (int off = 32; off > 0; off >>= 1) {
    const float od = __shfl_xor(d, off, 64);
    const int oi = __shfl_xor(index, off, 64);
    const bool better = oi >= 0 && (index < 0 || (Sign > 0 ? od > d : od < d) || (od == d && oi < index));
    if (better) { d = od; index = oi; }
  }
  return index;
}
__device__ __forceinline__ int wave_total(int v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ int wave_before(int v) {  // exclusive sum over the lanes
  int x = v;
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (int(threadIdx.x) >= off) x += y;
  }
  return x - v;
}

// ---------------------------------------------------------------------------------------------
// graph: owners, global edges, degrees, components (root = least vertex index) (post.cu:45-67)

// The last group whose offset is <= i (empty groups share offsets with the next one).
__device__ __forceinline__ int owner_of(const long long *off, int groups, long long i) {
  int lo = 0, hi = groups;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ int uf_root(int *up, int v) {
  int cur = ld_i(up + v);
  if (cur != v) {
    int prev = v, next;
    while (cur > (next = ld_i(up + cur))) {
      st_i(up + prev, next);  // path halving: a pointer only ever moves closer to its root
      prev = cur;
      cur = next;
    }
  }
  return cur;
}

__device__ __forceinline__ void uf_join(int *up, int a, int b) {
  int ra = uf_root(up, a), rb = uf_root(up, b);
  while (ra != rb) {
    const int lo = min(ra, rb), hi = max(ra, rb);
    const int seen = atomicCAS(up + hi, hi, lo);
    if (seen == hi) return;
    if (hi == ra) ra = uf_root(up, seen);
    else rb = uf_root(up, seen);
  }
}

__global__ void graph_vertices(const long long *voff, int k, int n, int *vlabel, int *root, int *degree) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  vlabel[i] = owner_of(voff, k, i);
  root[i] = i;
  degree[i] = 0;
}

// root: null when the components are not asked for.
__global__ void graph_edges(const unsigned *local, int m, const long long *voff, const long long *eoff, int k, int *elabel,
                            int2 *e, int *root, int *degree, int *bad) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m) return;
  const int l = owner_of(eoff, k, i);
  elabel[i] = l;
  const long long size = voff[l + 1] - voff[l];
  const unsigned a = local[2LL * i], b = local[2LL * i + 1];
  if ((long long)a >= size || (long long)b >= size) {
    atomicOr(bad, 1);
    e[i] = make_int2(0, 0);
    return;
  }
  const int ga = int(voff[l] + a), gb = int(voff[l] + b);
  e[i] = make_int2(ga, gb);
  atomicAdd(degree + ga, 1);
  atomicAdd(degree + gb, 1);
  if (root) uf_join(root, ga, gb);
}

__global__ void graph_flatten(int *root, int n) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  int r = ld_i(root + i), next;
  while (r != (next = ld_i(root + r))) r = next;  // read-only walk: a racing writer only stores roots
  st_i(root + i, r);
}

struct Graph {
  int n = 0, m = 0, k = 0;
  Buffer<long long> voff, eoff;
  Buffer<int> vlabel, elabel, root, degree;
  Buffer<int2> e;
};

// components: false leaves g.root as it is (each vertex its own).
Graph build_graph(Context &ctx, const DevicePacked &p, bool components = true) {
  const size_t k = p.labels.size();
  const bool ok = p.voff.size() == k + 1 && p.eoff.size() == k + 1 && p.voff.front() == 0 && p.eoff.front() == 0 &&
                  std::is_sorted(p.voff.begin(), p.voff.end()) && std::is_sorted(p.eoff.begin(), p.eoff.end()) &&
                  p.vertices.size() >= size_t(3 * p.n()) && p.radii.size() >= size_t(p.n()) &&
                  p.edges.size() >= size_t(2 * p.m());
  if (!ok) throw std::invalid_argument("invalid packed graph");
  if (p.n() > INT32_MAX || p.m() > INT32_MAX || k > size_t(INT32_MAX))
    throw std::invalid_argument("packed graph exceeds int32 work capacity");
  Graph g;
  g.n = int(p.n());
  g.m = int(p.m());
  g.k = int(k);
  g.voff = Buffer<long long>(ctx, k + 1);
  g.eoff = Buffer<long long>(ctx, k + 1);
  g.voff.upload(ctx, reinterpret_cast<const long long *>(p.voff.data()), k + 1);
  g.eoff.upload(ctx, reinterpret_cast<const long long *>(p.eoff.data()), k + 1);
  g.vlabel = Buffer<int>(ctx, std::max(g.n, 1));
  g.root = Buffer<int>(ctx, std::max(g.n, 1));
  g.degree = Buffer<int>(ctx, std::max(g.n, 1));
  g.elabel = Buffer<int>(ctx, std::max(g.m, 1));
  g.e = Buffer<int2>(ctx, std::max(g.m, 1));
  Buffer<int> bad(ctx, 1);
  bad.clear(ctx);
  auto s = ctx.stream();
  if (g.n) graph_vertices<<<grid(g.n), kThreads, 0, s>>>(g.voff.data(), g.k, g.n, g.vlabel.data(), g.root.data(), g.degree.data());
  if (g.m)
    graph_edges<<<grid(g.m), kThreads, 0, s>>>(p.edges.data(), g.m, g.voff.data(), g.eoff.data(), g.k, g.elabel.data(),
                                               g.e.data(), components ? g.root.data() : nullptr, g.degree.data(), bad.data());
  if (g.n && components) graph_flatten<<<grid(g.n), kThreads, 0, s>>>(g.root.data(), g.n);
  BROOK_LAUNCHED();
  if (read_one(ctx, bad.data())) throw std::invalid_argument("packed edge is out of bounds");
  return g;
}

// ---------------------------------------------------------------------------------------------
// selections (post.cu:70-117, 388-404)

__global__ void edge_both_kept(const int2 *e, int m, const int *keep, int *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < m) out[i] = keep[e[i].x] && keep[e[i].y];
}

__global__ void gather_offsets(const int *pos, const long long *off, int k, long long *out) {
  const int g = blockIdx.x * kThreads + threadIdx.x;
  if (g <= k) out[g] = pos[off[g]];
}

__global__ void scatter_vertices(const float *v, const float *r, const int *keep, const int *pos, int n, float *vout,
                                 float *rout) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n || !keep[i]) return;
  const int j = pos[i];
  vout[3LL * j] = v[3LL * i];
  vout[3LL * j + 1] = v[3LL * i + 1];
  vout[3LL * j + 2] = v[3LL * i + 2];
  rout[j] = r[i];
}

__global__ void scatter_edges(const int2 *e, const int *elabel, const int *ekeep, const int *epos, const int *vpos,
                              const long long *new_voff, int m, unsigned *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m || !ekeep[i]) return;
  const long long base = new_voff[elabel[i]];
  const int j = epos[i];
  out[2LL * j] = unsigned(vpos[e[i].x] - base);
  out[2LL * j + 1] = unsigned(vpos[e[i].y] - base);
}

__global__ void copy_edge_rows(const unsigned *in, const int *keep, const int *pos, int m, unsigned *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m || !keep[i]) return;
  out[2LL * pos[i]] = in[2LL * i];
  out[2LL * pos[i] + 1] = in[2LL * i + 1];
}

// Exclusive positions of `flags` (n + 1 entries, the last the total) and the per-group offsets
// they give at the group boundaries `off`.
std::vector<int64_t> positions(Context &ctx, const Buffer<int> &flags, int n, const Buffer<long long> &off, int k,
                               Buffer<int> &pos, Buffer<long long> &new_off) {
  Buffer<int> padded(ctx, size_t(n) + 1);
  if (n) BROOK_HIP(hipMemcpyAsync(padded.data(), flags.data(), size_t(n) * 4, hipMemcpyDeviceToDevice, ctx.stream()));
  BROOK_HIP(hipMemsetAsync(padded.data() + n, 0, 4, ctx.stream()));
  pos = Buffer<int>(ctx, size_t(n) + 1);
  exclusive_sum(ctx, padded.data(), pos.data(), n + 1);
  new_off = Buffer<long long>(ctx, size_t(k) + 1);
  gather_offsets<<<grid(k + 1), kThreads, 0, ctx.stream()>>>(pos.data(), off.data(), k, new_off.data());
  BROOK_LAUNCHED();
  std::vector<long long> h = new_off.download(ctx);
  return std::vector<int64_t>(h.begin(), h.end());
}

// The kept vertices in order and the edges with both ends kept, in order (post.cu:86-109).
DevicePacked select_vertices(Context &ctx, const DevicePacked &p, const Buffer<int> &keep, const Graph &g) {
  DevicePacked out;
  out.labels = p.labels;
  out.anisotropy = p.anisotropy;
  Buffer<int> vpos, epos, ekeep(ctx, std::max(g.m, 1));
  Buffer<long long> new_voff, new_eoff;
  out.voff = positions(ctx, keep, g.n, g.voff, g.k, vpos, new_voff);
  if (g.m) edge_both_kept<<<grid(g.m), kThreads, 0, ctx.stream()>>>(g.e.data(), g.m, keep.data(), ekeep.data());
  BROOK_LAUNCHED();
  out.eoff = positions(ctx, ekeep, g.m, g.eoff, g.k, epos, new_eoff);
  out.vertices = Buffer<float>(ctx, size_t(std::max<int64_t>(3 * out.n(), 1)));
  out.radii = Buffer<float>(ctx, size_t(std::max<int64_t>(out.n(), 1)));
  out.edges = Buffer<uint32_t>(ctx, size_t(std::max<int64_t>(2 * out.m(), 1)));
  if (g.n)
    scatter_vertices<<<grid(g.n), kThreads, 0, ctx.stream()>>>(p.vertices.data(), p.radii.data(), keep.data(), vpos.data(),
                                                               g.n, out.vertices.data(), out.radii.data());
  if (g.m)
    scatter_edges<<<grid(g.m), kThreads, 0, ctx.stream()>>>(g.e.data(), g.elabel.data(), ekeep.data(), epos.data(),
                                                            vpos.data(), new_voff.data(), g.m, out.edges.data());
  BROOK_LAUNCHED();
  return out;
}

// The edges with keep[i] in order; vertices unchanged (post.cu:388-404).
DevicePacked select_edges(Context &ctx, DevicePacked p, const Buffer<int> &keep, const Graph &g) {
  Buffer<int> epos;
  Buffer<long long> new_eoff;
  p.eoff = positions(ctx, keep, g.m, g.eoff, g.k, epos, new_eoff);
  Buffer<uint32_t> edges(ctx, size_t(std::max<int64_t>(2 * p.m(), 1)));
  if (g.m) copy_edge_rows<<<grid(g.m), kThreads, 0, ctx.stream()>>>(p.edges.data(), keep.data(), epos.data(), g.m, edges.data());
  BROOK_LAUNCHED();
  p.edges = std::move(edges);
  return p;
}

// ---------------------------------------------------------------------------------------------
// sorted unique edge keys -> local edges (post.cu:273-292)

__global__ void unique_heads(const unsigned long long *keys, int n, int *flags) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) flags[i] = keys[i] != kNone && (i == 0 || keys[i] != keys[i - 1]);
}

__global__ void compact_keys(const unsigned long long *keys, const int *flags, const int *pos, int n,
                             unsigned long long *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n && flags[i]) out[pos[i]] = keys[i];
}

// Per group: the first unique key whose lower end is at or past the group's first vertex.
__global__ void key_offsets(const unsigned long long *keys, int n, const long long *voff, int k, long long *eoff) {
  const int g = blockIdx.x * kThreads + threadIdx.x;
  if (g > k) return;
  const unsigned long long target = (unsigned long long)voff[g] << 32;
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (keys[mid] < target) lo = mid + 1;
    else hi = mid;
  }
  eoff[g] = lo;
}

__global__ void local_pairs(const unsigned long long *keys, int n, const int *vlabel, const long long *voff, unsigned *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const unsigned a = unsigned(keys[i] >> 32), b = unsigned(keys[i]);
  const long long base = voff[vlabel[a]];
  out[2LL * i] = unsigned(a - base);
  out[2LL * i + 1] = unsigned(b - base);
}

DevicePacked edges_from_keys(Context &ctx, DevicePacked p, const Graph &g, Buffer<unsigned long long> &keys, int count) {
  Buffer<unsigned char> scratch;
  Buffer<unsigned long long> sorted(ctx, std::max(count, 1));
  if (count)
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortKeys(t, b, keys.data(), sorted.data(), count, 0, 64, ctx.stream());
    });
  Buffer<int> flags(ctx, std::max(count, 1)), pos(ctx, std::max(count, 1));
  int total = 0;
  Buffer<unsigned long long> unique(ctx, std::max(count, 1));
  if (count) {
    unique_heads<<<grid(count), kThreads, 0, ctx.stream()>>>(sorted.data(), count, flags.data());
    exclusive_sum(ctx, flags.data(), pos.data(), count);
    compact_keys<<<grid(count), kThreads, 0, ctx.stream()>>>(sorted.data(), flags.data(), pos.data(), count, unique.data());
    BROOK_LAUNCHED();
    total = read_one(ctx, pos.data() + count - 1) + read_one(ctx, flags.data() + count - 1);
  }
  Buffer<long long> eoff(ctx, size_t(g.k) + 1);
  key_offsets<<<grid(g.k + 1), kThreads, 0, ctx.stream()>>>(unique.data(), total, g.voff.data(), g.k, eoff.data());
  Buffer<uint32_t> edges(ctx, size_t(std::max(2 * total, 1)));
  if (total) local_pairs<<<grid(total), kThreads, 0, ctx.stream()>>>(unique.data(), total, g.vlabel.data(), g.voff.data(), edges.data());
  BROOK_LAUNCHED();
  std::vector<long long> h = eoff.download(ctx);
  p.eoff.assign(h.begin(), h.end());
  p.edges = std::move(edges);
  return p;
}

// ---------------------------------------------------------------------------------------------
// prune_unused (post.cu:433-442)

__global__ void nonzero(const int *degree, int n, int *keep, int *zero) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  keep[i] = degree[i] != 0;
  if (!degree[i]) atomicOr(zero, 1);
}

DevicePacked prune_unused(Context &ctx, DevicePacked p) {
  Graph g = build_graph(ctx, p, false);
  if (!g.n) return p;
  Buffer<int> keep(ctx, g.n), zero(ctx, 1);
  zero.clear(ctx);
  nonzero<<<grid(g.n), kThreads, 0, ctx.stream()>>>(g.degree.data(), g.n, keep.data(), zero.data());
  BROOK_LAUNCHED();
  if (!read_one(ctx, zero.data())) return p;
  return select_vertices(ctx, p, keep, g);
}

// ---------------------------------------------------------------------------------------------
// remove_dust (post.cu:115-137, 443-475)

__global__ void edge_lengths(const float *v, const int2 *e, const int *root, int m, double *total, int *count) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m) return;
  const int a = e[i].x, b = e[i].y;
  const double x = double(v[3LL * b] - v[3LL * a]), y = double(v[3LL * b + 1] - v[3LL * a + 1]),
               z = double(v[3LL * b + 2] - v[3LL * a + 2]);
  const int r = root[a];
  atomicAdd(total + r, sqrt((x * x + y * y) + z * z));
  atomicAdd(count + r, 1);
}

// Keep a root whose double total clears the threshold; a root within count * 2^-23 * threshold
// of it is marked undecided (2) for the float32 pairwise rule.
__global__ void dust_decide(const double *total, const int *count, int n, double threshold, int *keep_root) {
  const int r = blockIdx.x * kThreads + threadIdx.x;
  if (r >= n) return;
  const bool near = count[r] > 0 && fabs(total[r] - threshold) <= count[r] * (1.0 / 8388608.0) * threshold;
  keep_root[r] = near ? 2 : (total[r] > threshold ? 1 : 0);
}

__device__ __forceinline__ float length32(const float *v, int a, int b) {
  float x = v[3LL * b] - v[3LL * a], y = v[3LL * b + 1] - v[3LL * a + 1], z = v[3LL * b + 2] - v[3LL * a + 2];
  x = x * x;
  y = y * y;
  z = z * z;
  return sqrtf((x + y) + z);
}

// NumPy's pairwise float32 sum (numpy loops_utils pairwise_sum, block 128, eight partial sums)
// over the lengths of `count` edges listed at `list`, without recursion: the split tree is
// walked depth first, left before right, with partial sums on an explicit stack.
__device__ float pairwise_lengths(const float *v, const int2 *e, const int *list, int count) {
  struct Frame { int start, n, state; float left; };
  Frame st[40];
  int sp = 0;
  st[sp++] = Frame{0, count, 0, 0.0f};
  float result = 0.0f;
  while (sp) {
    Frame &f = st[sp - 1];
    if (f.n <= 128) {
      float s;
      if (f.n < 8) {
        s = -0.0f;
        for (int i = 0; i < f.n; ++i) s += length32(v, e[list[f.start + i]].x, e[list[f.start + i]].y);
      } else {
        float r[8];
        for (int j = 0; j < 8; ++j) r[j] = length32(v, e[list[f.start + j]].x, e[list[f.start + j]].y);
        int i = 8;
        for (; i + 8 <= f.n; i += 8)
          for (int j = 0; j < 8; ++j) r[j] += length32(v, e[list[f.start + i + j]].x, e[list[f.start + i + j]].y);
        s = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
        for (; i < f.n; ++i) s += length32(v, e[list[f.start + i]].x, e[list[f.start + i]].y);
      }
      --sp;
      if (!sp) { result = s; break; }
      Frame &up = st[sp - 1];  // a finished half returns to its parent
      if (up.state == 1) up.left = s, up.state = 2;
      else up.left = up.left + s, up.state = 3;
      continue;
    }
    int half = f.n / 2;
    half -= half % 8;
    if (f.state == 0) {
      f.state = 1;
      st[sp++] = Frame{f.start, half, 0, 0.0f};
    } else if (f.state == 2) {
      st[sp++] = Frame{f.start + half, f.n - half, 0, 0.0f};
    } else {  // both halves done
      const float s = f.left;
      --sp;
      if (!sp) { result = s; break; }
      Frame &up = st[sp - 1];
      if (up.state == 1) up.left = s, up.state = 2;
      else up.left = up.left + s, up.state = 3;
    }
  }
  return result;
}

// One lane per undecided root: its edges in edge order (list segment) under the float32 rule.
__global__ void dust_pairwise(const float *v, const int2 *e, const int *roots, const int *list, const long long *seg, int count,
                              double threshold, int *keep_root) {
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= count) return;
  const float s = pairwise_lengths(v, e, list + seg[c], int(seg[c + 1] - seg[c]));
  keep_root[roots[c]] = double(s) > threshold ? 1 : 0;
}

__global__ void undecided_keys(const int2 *e, const int *root, const int *slot, int m, int sentinel, int *key, int *index) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m) return;
  const int s = slot[root[e[i].x]];
  key[i] = s >= 0 ? s : sentinel;
  index[i] = i;
}

__global__ void undecided_slots(const int *keep_root, const int *pos, int n, int *slot, int *roots) {
  const int r = blockIdx.x * kThreads + threadIdx.x;
  if (r >= n) return;
  slot[r] = keep_root[r] == 2 ? pos[r] : -1;
  if (keep_root[r] == 2) roots[pos[r]] = r;
}

__global__ void is_two(const int *keep_root, int n, int *out) {
  const int r = blockIdx.x * kThreads + threadIdx.x;
  if (r < n) out[r] = keep_root[r] == 2;
}

__global__ void broadcast_root(const int *keep_root, const int *root, int n, int *keep) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) keep[i] = keep_root[root[i]];
}

__global__ void count_per_slot(const int *key, int m, int count, int *per) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < m && key[i] < count) atomicAdd(per + key[i], 1);
}

DevicePacked remove_dust(Context &ctx, DevicePacked p, double threshold) {
  if (threshold == 0 || p.n() == 0) return p;
  Graph g = build_graph(ctx, p);
  auto s = ctx.stream();
  Buffer<double> total(ctx, g.n);
  Buffer<int> count(ctx, g.n), keep_root(ctx, g.n);
  total.clear(ctx);
  count.clear(ctx);
  if (g.m) edge_lengths<<<grid(g.m), kThreads, 0, s>>>(p.vertices.data(), g.e.data(), g.root.data(), g.m, total.data(), count.data());
  dust_decide<<<grid(g.n), kThreads, 0, s>>>(total.data(), count.data(), g.n, threshold, keep_root.data());
  BROOK_LAUNCHED();
  // undecided roots: their edges grouped by root in edge order (a stable sort by slot)
  Buffer<int> two(ctx, g.n + 1), pos(ctx, g.n + 1);
  is_two<<<grid(g.n), kThreads, 0, s>>>(keep_root.data(), g.n, two.data());
  BROOK_HIP(hipMemsetAsync(two.data() + g.n, 0, 4, s));
  exclusive_sum(ctx, two.data(), pos.data(), g.n + 1);
  const int undecided = read_one(ctx, pos.data() + g.n);
  if (undecided) {
    Buffer<int> slot(ctx, g.n), roots(ctx, undecided);
    undecided_slots<<<grid(g.n), kThreads, 0, s>>>(keep_root.data(), pos.data(), g.n, slot.data(), roots.data());
    Buffer<int> key(ctx, g.m), key_sorted(ctx, g.m), index(ctx, g.m), list(ctx, g.m);
    undecided_keys<<<grid(g.m), kThreads, 0, s>>>(g.e.data(), g.root.data(), slot.data(), g.m, undecided, key.data(), index.data());
    BROOK_LAUNCHED();
    Buffer<unsigned char> scratch;
    int bits = 1;
    while ((1LL << bits) <= undecided) ++bits;
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortPairs(t, b, key.data(), key_sorted.data(), index.data(), list.data(), g.m, 0, bits, s);
    });
    Buffer<int> per(ctx, undecided + 1);
    per.clear(ctx);
    count_per_slot<<<grid(g.m), kThreads, 0, s>>>(key.data(), g.m, undecided, per.data());
    BROOK_LAUNCHED();
    std::vector<int> h = per.download(ctx);
    std::vector<long long> seg(size_t(undecided) + 1, 0);
    for (int c = 0; c < undecided; ++c) seg[c + 1] = seg[c] + h[c];
    Buffer<long long> seg_dev(ctx, seg.size());
    seg_dev.upload(ctx, seg.data(), seg.size());
    dust_pairwise<<<grid(undecided), kThreads, 0, s>>>(p.vertices.data(), g.e.data(), roots.data(), list.data(), seg_dev.data(),
                                                       undecided, threshold, keep_root.data());
    BROOK_LAUNCHED();
  }
  Buffer<int> keep(ctx, g.n);
  broadcast_root<<<grid(g.n), kThreads, 0, s>>>(keep_root.data(), g.root.data(), g.n, keep.data());
  BROOK_LAUNCHED();
  return select_vertices(ctx, p, keep, g);
}

// ---------------------------------------------------------------------------------------------
// Components taking part in a sequential rule: their vertices (ascending index) and edges (edge
// order) as contiguous segments in slot order, local ids = position in the segment.

// Adds 1 to count[slot] for every lane with `on` (all lanes of the wave here): lanes of consecutive
// equal slots add together, so a long run of one component is one atomic per wave.
__device__ __forceinline__ void count_runs(int *count, int slot, bool on) {
  const int lane = int(threadIdx.x) & 63;
  const int key = on ? slot : -1, before = __shfl_up(key, 1, 64);
  const unsigned long long heads = __builtin_amdgcn_ballot_w64(lane == 0 || key != before);
  if (!on || !((heads >> lane) & 1ULL)) return;
  const unsigned long long after = lane == 63 ? 0ULL : heads >> (lane + 1);
  atomicAdd(count + slot, after ? __ffsll((long long)after) : 64 - lane);
}

// critical: vertices of degree 1 or at least 3; branch: a vertex of degree at least 3.
__global__ void component_sizes(const int *root, const int *degree, int n, const int2 *e, int m, int *nv, int *ne, int *branch,
                                int *critical) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int r = i < n ? root[i] : 0, d = i < n ? degree[i] : 0;
  count_runs(nv, r, i < n);
  count_runs(critical, r, d == 1 || d >= 3);
  if (d >= 3) branch[r] = 1;
  count_runs(ne, i < m ? root[e[i].x] : 0, i < m);
}

__global__ void pick_components(const int *nv, const int *ne, const int *branch, int n, bool trees, int *flag) {
  const int r = blockIdx.x * kThreads + threadIdx.x;
  if (r >= n) return;
  flag[r] = trees ? (branch[r] && ne[r] == nv[r] - 1) : (ne[r] > 0 && ne[r] - nv[r] + 1 > 0);
}

__global__ void component_slots(const int *flag, const int *pos, const int *nv, const int *ne, const int *critical, int n,
                                int *slot, int3 *sizes) {
  const int r = blockIdx.x * kThreads + threadIdx.x;
  if (r >= n) return;
  slot[r] = flag[r] ? pos[r] : -1;
  if (flag[r]) {
    sizes[pos[r]] = make_int3(nv[r], ne[r], critical[r]);
  }
}

__global__ void slot_keys_vertices(const int *root, const int *slot, int n, int sentinel, int *key, int *index) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const int s = slot[root[i]];
  key[i] = s >= 0 ? s : sentinel;
  index[i] = i;
}

__global__ void slot_keys_edges(const int2 *e, const int *root, const int *slot, int m, int sentinel, int *key, int *index) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m) return;
  const int s = slot[root[e[i].x]];
  key[i] = s >= 0 ? s : sentinel;
  index[i] = i;
}

__global__ void local_ids(const int *vlist, const int *root, const int *slot, const long long *vs, int count, int *local) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j >= count) return;
  const int v = vlist[j];
  local[v] = int(j - vs[slot[root[v]]]);
}

__global__ void local_rows(const int *elist, const int2 *e, const int *local, int count, int2 *rows) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j >= count) return;
  const int2 ge = e[elist[j]];
  rows[j] = make_int2(local[ge.x], local[ge.y]);
}

struct Pieces {
  int count = 0, nv = 0, ne = 0;  // components, their vertices and edges
  Buffer<int> slot;               // per root: slot or -1
  Buffer<int> vlist, elist;       // global ids in slot order
  Buffer<long long> vs, es;       // per slot: segment starts (count + 1)
  std::vector<long long> vs_host, es_host;
  std::vector<int> critical;      // per slot: vertices of degree 1 or at least 3
  Buffer<int> local;              // per vertex of a piece: local id
  Buffer<int2> rows;              // per edge of a piece: local (x, y) as stored
  Buffer<int> comp_of_edge;       // per edge of a piece: its component
};

// The components (of `count`) whose state fits LDS and the others, as lists on the device;
// lds: the largest fitting state, which every block of the launch asks for, so one large component
// leaves the small ones fewer waves: the loops of 20 000 components of 14 vertices take 2.0 ms, beside one
// of 2500 vertices 8.6 (a lane per component 2.1 and 15.3).
struct Split {
  Buffer<int> small, large;
  int nsmall = 0, nlarge = 0;
  size_t lds = 0;
};
template <class Bytes> Split split_pieces(Context &ctx, const Pieces &pc, Bytes &&bytes) {
  Split sp;
  std::vector<int> small, large;
  for (int c = 0; c < pc.count; ++c) {
    const long long nv = pc.vs_host[size_t(c) + 1] - pc.vs_host[size_t(c)], E = pc.es_host[size_t(c) + 1] - pc.es_host[size_t(c)];
    const size_t need = bytes(size_t(c), size_t(nv), size_t(E));
    // 16-bit indices: entries are numbered up to 2 E + 4
    if (need <= kLdsPiece && 2 * E + 4 < 32768 && nv < 32768) {
      small.push_back(c);
      sp.lds = std::max(sp.lds, need);
    } else {
      large.push_back(c);
    }
  }
  sp.nsmall = int(small.size());
  sp.nlarge = int(large.size());
  sp.small = Buffer<int>(ctx, std::max<size_t>(small.size(), 1));
  sp.large = Buffer<int>(ctx, std::max<size_t>(large.size(), 1));
  if (sp.nsmall) sp.small.upload(ctx, small.data(), small.size());
  if (sp.nlarge) sp.large.upload(ctx, large.data(), large.size());
  return sp;
}

Pieces pieces_of(Context &ctx, const Graph &g, bool trees) {
  Pieces pc;
  auto s = ctx.stream();
  Buffer<int> sums(ctx, size_t(4) * g.n), flag(ctx, g.n + 1), pos(ctx, g.n + 1);
  sums.clear(ctx);
  int *nv = sums.data(), *ne = nv + g.n, *branch = ne + g.n, *critical = branch + g.n;
  component_sizes<<<grid(std::max(g.n, g.m)), kThreads, 0, s>>>(g.root.data(), g.degree.data(), g.n, g.e.data(), g.m, nv, ne,
                                                               branch, critical);
  pick_components<<<grid(g.n), kThreads, 0, s>>>(nv, ne, branch, g.n, trees, flag.data());
  BROOK_LAUNCHED();
  BROOK_HIP(hipMemsetAsync(flag.data() + g.n, 0, 4, s));
  exclusive_sum(ctx, flag.data(), pos.data(), g.n + 1);
  pc.count = read_one(ctx, pos.data() + g.n);
  if (!pc.count) return pc;
  pc.slot = Buffer<int>(ctx, g.n);
  Buffer<int3> sizes(ctx, pc.count);
  component_slots<<<grid(g.n), kThreads, 0, s>>>(flag.data(), pos.data(), nv, ne, critical, g.n, pc.slot.data(), sizes.data());
  BROOK_LAUNCHED();
  const std::vector<int3> h = sizes.download(ctx);
  pc.vs_host.assign(1, 0);
  pc.es_host.assign(1, 0);
  for (const int3 &c : h) {
    pc.vs_host.push_back(pc.vs_host.back() + c.x);
    pc.es_host.push_back(pc.es_host.back() + c.y);
    pc.critical.push_back(c.z);
  }
  pc.nv = int(pc.vs_host.back());
  pc.ne = int(pc.es_host.back());
  pc.vs = Buffer<long long>(ctx, pc.vs_host.size());
  pc.es = Buffer<long long>(ctx, pc.es_host.size());
  pc.vs.upload(ctx, pc.vs_host.data(), pc.vs_host.size());
  pc.es.upload(ctx, pc.es_host.data(), pc.es_host.size());
  int bits = 1;
  while ((1LL << bits) <= pc.count) ++bits;
  Buffer<unsigned char> scratch;
  {  // vertices by (slot, index): a stable sort by slot; the other vertices sort last
    Buffer<int> key(ctx, g.n), key_sorted(ctx, g.n), index(ctx, g.n);
    pc.vlist = Buffer<int>(ctx, g.n);
    slot_keys_vertices<<<grid(g.n), kThreads, 0, s>>>(g.root.data(), pc.slot.data(), g.n, pc.count, key.data(), index.data());
    BROOK_LAUNCHED();
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortPairs(t, b, key.data(), key_sorted.data(), index.data(), pc.vlist.data(), g.n, 0, bits, s);
    });
  }
  {
    Buffer<int> key(ctx, g.m), index(ctx, g.m);
    pc.elist = Buffer<int>(ctx, g.m);
    pc.comp_of_edge = Buffer<int>(ctx, g.m);  // the sorted keys
    slot_keys_edges<<<grid(g.m), kThreads, 0, s>>>(g.e.data(), g.root.data(), pc.slot.data(), g.m, pc.count, key.data(),
                                                   index.data());
    BROOK_LAUNCHED();
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortPairs(t, b, key.data(), pc.comp_of_edge.data(), index.data(), pc.elist.data(), g.m, 0, bits, s);
    });
  }
  pc.local = Buffer<int>(ctx, g.n);
  pc.rows = Buffer<int2>(ctx, std::max(pc.ne, 1));
  local_ids<<<grid(pc.nv), kThreads, 0, s>>>(pc.vlist.data(), g.root.data(), pc.slot.data(), pc.vs.data(), pc.nv, pc.local.data());
  if (pc.ne) local_rows<<<grid(pc.ne), kThreads, 0, s>>>(pc.elist.data(), g.e.data(), pc.local.data(), pc.ne, pc.rows.data());
  BROOK_LAUNCHED();
  return pc;
}

// ---------------------------------------------------------------------------------------------
// remove_loops: one wave per cyclic component (post_kernels.cuh:22-199)

// A component's state: I indexes (pointer to short in LDS, int in device memory), B bytes.
template <class I, class B> struct LoopState {
  I rx, ry;                       // 2 E + 2 rows: (x, y), x = -1 once dead
  I nbr, nxt, prv, rid, mul;      // 2 E + 4 list entries
  I head, tail, cnt, seen, order;  // nv + 1
  I branch, path;                 // nv + 1
  I node, parent, depth;          // 2 E + 2: the search stack
  B drop;                         // nv + 1
  int freelist, bump, entry_cap;
  int nrows;
  long long nlive;
  bool overflow;  // the entry pool ran out (only rows repeated in both orientations can do that)

  __device__ int find(int a, int b) const {
    for (int e = head[a]; e >= 0; e = nxt[e])
      if (nbr[e] == b) return e;
    return -1;
  }
  __device__ int entry() {
    if (freelist >= 0) { const int e = freelist; freelist = nxt[e]; return e; }
    if (bump == entry_cap) { overflow = true; return entry_cap - 1; }  // in bounds; the result is discarded
    return bump++;
  }
  __device__ void link(int a, int b, int r) {
    const int e = entry();
    nbr[e] = b;
    rid[e] = r;
    mul[e] = 1;
    nxt[e] = -1;
    prv[e] = tail[a];
    if (tail[a] >= 0) nxt[tail[a]] = e;
    else head[a] = e;
    tail[a] = e;
  }
  __device__ void unlink(int a, int e) {
    if (prv[e] >= 0) nxt[prv[e]] = nxt[e];
    else head[a] = nxt[e];
    if (nxt[e] >= 0) prv[nxt[e]] = prv[e];
    else tail[a] = prv[e];
    nxt[e] = freelist;
    freelist = e;
  }
  __device__ void add_row(int x, int y) {
    const int r = nrows++;
    rx[r] = x;
    ry[r] = y;
    nlive++;
    cnt[x] += 1;
    cnt[y] += 1;
    const int f = find(x, y);
    if (f >= 0) {  // a repeated pair: the first match of each list counts it
      mul[f] += 1;
      const int back = find(y, x);
      mul[back] += 1;
    } else {
      link(x, y, r);
      link(y, x, r);
    }
  }
};

// The arrays of a component laid out one after another: index arrays of T, then bytes.
template <class T> size_t loop_bytes(size_t nv, size_t E) {
  return sizeof(T) * (2 * (2 * E + 2) + 5 * (2 * E + 4) + 7 * (nv + 1) + 3 * (2 * E + 2)) + (nv + 1);
}
template <class I, class B> __device__ LoopState<I, B> loop_state(I at, int nv, int E) {
  LoopState<I, B> s;
  auto take = [&](int n) { I p = at; at += n; return p; };
  s.node = take(2 * E + 2);  // first: the list build counts in its place, in 32 bits
  s.parent = take(2 * E + 2);
  s.depth = take(2 * E + 2);
  s.rx = take(2 * E + 2);
  s.ry = take(2 * E + 2);
  s.nbr = take(2 * E + 4);
  s.nxt = take(2 * E + 4);
  s.prv = take(2 * E + 4);
  s.rid = take(2 * E + 4);
  s.mul = take(2 * E + 4);
  s.head = take(nv + 1);
  s.tail = take(nv + 1);
  s.cnt = take(nv + 1);
  s.seen = take(nv + 1);
  s.order = take(nv + 1);
  s.branch = take(nv + 1);
  s.path = take(nv + 1);
  s.drop = (B)at;
  s.freelist = -1;
  s.bump = 2 * E;
  s.entry_cap = 2 * E + 4;
  s.nrows = E;
  s.nlive = E;
  s.overflow = false;
  return s;
}

// The neighbour lists of the input rows, as add_row row by row gives them: counted, given out and put
// in row order per vertex by lanes of their own. W: 32-bit counters (the stack's place: a cyclic
// component has at least as many rows as vertices, so 6 E + 6 16-bit slots hold nv of them).
template <class W, class I, class B>
__device__ void loop_lists(LoopState<I, B> &s, W counter, int nv, int E, const int2 *rows_in) {
  const int lane = threadIdx.x;
  for (int v = lane; v < nv; v += 64) counter[v] = 0;
  wave_sync();
  for (int r = lane; r < E; r += 64) {
    const int2 x = rows_in[r];
    s.rx[r] = x.x;
    s.ry[r] = x.y;
    __hip_atomic_fetch_add(counter + x.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(counter + x.y, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  wave_sync();
  int base = 0;
  for (int v0 = 0; v0 < nv; v0 += 64) {  // segment starts: head for now
    const int v = v0 + lane, c = v < nv ? counter[v] : 0, before = wave_before(c);
    if (v < nv) {
      s.cnt[v] = c;
      s.head[v] = base + before;
      s.seen[v] = 0;
      counter[v] = base + before;
    }
    base += wave_total(c);
  }
  wave_sync();
  for (int r = lane; r < E; r += 64) {
    const int x = s.rx[r], y = s.ry[r];
    const int a = __hip_atomic_fetch_add(counter + x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    s.rid[a] = r;
    const int b = __hip_atomic_fetch_add(counter + y, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    s.rid[b] = r;
  }
  wave_sync();
  bool dropped = false;
  for (int v = lane; v < nv; v += 64) {
    const int e0 = s.head[v], e1 = e0 + s.cnt[v];
    for (int i = e0 + 1; i < e1; ++i) {  // by row
      const int r = s.rid[i];
      int j = i - 1;
      while (j >= e0 && s.rid[j] > r) { s.rid[j + 1] = s.rid[j]; --j; }
      s.rid[j + 1] = r;
    }
    int head = -1, tail = -1;
    for (int i = e0; i < e1; ++i) {
      const int r = s.rid[i], x = s.rx[r], y = s.ry[r], other = x == v ? y : x;
      int first = -1;  // an earlier row's entry of the same pair
      for (int f = head; f >= 0; f = s.nxt[f])
        if (s.nbr[f] == other && s.rid[f] != r) { first = f; break; }
      if (first >= 0) {
        s.mul[first] += 1;
        s.rid[i] = -2;  // a free entry
        dropped = true;
        continue;
      }
      s.nbr[i] = other;
      s.mul[i] = 1;
      s.nxt[i] = -1;
      s.prv[i] = tail;
      if (tail >= 0) s.nxt[tail] = i;
      else head = i;
      tail = i;
    }
    s.head[v] = head;
    s.tail[v] = tail;
  }
  wave_sync();
  if (__builtin_amdgcn_ballot_w64(dropped))
    for (int i = 0; i < 2 * E; ++i)
      if (s.rid[i] == -2) { s.nxt[i] = s.freelist; s.freelist = i; }
}

__device__ __forceinline__ float sq_dist(const float *P, float x, float y, float z) {
  const float dx = P[0] - x, dy = P[1] - y, dz = P[2] - z;
  return (dx * dx + dy * dy) + dz * dz;
}

template <class I, class B>
__device__ void loops_component(LoopState<I, B> &s, int nv, int E, const int *vl, const float *vertices, const float *radii,
                                int2 *rows_out, int *ne_out, int *failed) {
  const int lane = threadIdx.x;
  const int row_cap = 2 * E + 2;
  auto P = [&](int v) { return vertices + 3LL * vl[v]; };
  auto fail = [&](int bit) { if (lane == 0) atomicOr(failed, bit); };
  int app0 = s.nrows, app1 = s.nrows;  // rows appended by the previous iteration
  int first = 0;                       // no row before it lives
  const long long budget = 64LL * (E + nv) + 64;
  for (long long iteration = 0;; ++iteration) {
    if (iteration > budget) { fail(1); break; }
    if (s.overflow) { fail(2); break; }
    if (s.nlive == 0) break;
    while (s.rx[first] < 0) first++;
    // depth-first search from the first live row's first end
    int sp = 0, plen = 0, node = -1, nseen = 0;
    bool found = false;
    s.node[sp] = s.rx[first];
    s.parent[sp] = -1;
    s.depth[sp++] = 0;
    while (sp) {
      --sp;
      node = s.node[sp];
      const int parent = s.parent[sp], depth = s.depth[sp];
      if (plen > depth) plen = depth;
      s.path[plen++] = node;
      if (s.seen[node]) { found = true; break; }
      s.seen[node] = 1;
      s.order[nseen++] = node;
      for (int e = s.head[node]; e >= 0; e = s.nxt[e]) {
        const int to = s.nbr[e];
        if (to == parent) continue;
        s.node[sp] = to;
        s.parent[sp] = node;
        s.depth[sp++] = depth + 1;
      }
    }
    wave_sync();
    for (int j = lane; j < nseen; j += 64) s.seen[s.order[j]] = 0;
    wave_sync();
    if (!found || plen <= 1) break;
    int i0 = 0;
    while (i0 < plen - 1 && s.path[i0] != node) i0++;
    if (plen - i0 < 3) break;
    const I cy = s.path + i0;
    const int cl = plen - i0;
    int nb = 0;
    for (int j = 0; j + 1 < cl; ++j)
      if (s.cnt[cy[j]] >= 3) s.branch[nb++] = cy[j];
    for (int i = 1; i < nb; ++i) {  // ascending (few)
      const int x = s.branch[i];
      int j = i - 1;
      while (j >= 0 && s.branch[j] > x) { s.branch[j + 1] = s.branch[j]; --j; }
      s.branch[j + 1] = x;
    }
    wave_sync();
    for (int j = lane; j < cl; j += 64) s.drop[j] = 0;
    wave_sync();
    int add_a = -1, add_b = -1, hub = -1;
    bool star = false, whole = false;  // whole: every edge of the cycle goes
    if (nb == 0) {
      whole = true;
    } else if (nb == 1) {
      // the farthest cycle node, the lower one on ties; a first node at a NaN distance stays
      const int bn = s.branch[0];
      const float bx = P(bn)[0], by = P(bn)[1], bz = P(bn)[2];
      float best = 0.0f;
      int end = -1;
      for (int j = lane; j + 1 < cl; j += 64) {
        const int v = cy[j];
        const float d = sq_dist(P(v), bx, by, bz);
        if (d == d && (end < 0 || d > best || (d == best && v < end))) { best = d; end = v; }
      }
      end = wave_extreme<1>(best, end);
      const float d0 = sq_dist(P(cy[0]), bx, by, bz);
      if (d0 != d0) end = cy[0];
      whole = true;
      add_a = bn;
      add_b = end;
    } else if (nb == 2) {
      const int L = cl - 1;
      int p0 = -1, p1 = -1;
      for (int j = 0; j < L; ++j)
        if (s.cnt[cy[j + 1]] >= 3) {
          if (p0 < 0) p0 = j;
          else p1 = j;
        }
      const bool inner = double(p1 - p0) < double(L) / 2.0;
      for (int j = lane; j + 1 < cl; j += 64) {
        const bool on_inner = j - 1 >= 0 && j - 1 >= p0 && j <= p1;
        if (!(inner ? on_inner : !on_inner)) s.drop[j] = 1;
      }
    } else {
      float cx = 0.0f, cyy = 0.0f, cz = 0.0f;
      for (int i = 0; i < nb; ++i) { const float *q = P(s.branch[i]); cx += q[0]; cyy += q[1]; cz += q[2]; }
      cx /= float(nb);
      cyy /= float(nb);
      cz /= float(nb);
      // the nearest vertex, the lowest on ties; a first vertex at a NaN distance stays
      float best = 0.0f;
      for (int v = lane; v < nv; v += 64) {
        const float d = sq_dist(P(v), cx, cyy, cz);
        if (d == d && (hub < 0 || d < best)) { best = d; hub = v; }
      }
      hub = wave_extreme<-1>(best, hub);
      const float d0 = sq_dist(P(0), cx, cyy, cz);
      if (d0 != d0) hub = 0;
      float far = 0.0f;
      for (int i = 0; i < nb; ++i) {
        const float d = sq_dist(P(s.branch[i]), P(hub)[0], P(hub)[1], P(hub)[2]);
        if (i == 0 || d > far) far = d;
      }
      if (sqrtf(far) > radii[vl[hub]]) {
        s.drop[0] = 1;
      } else {
        whole = star = true;
      }
    }
    wave_sync();
    for (int r = app0; r < app1; ++r) {
      const int x = s.rx[r], y = s.ry[r];
      if (x > y) { s.rx[r] = y; s.ry[r] = x; }
    }
    for (int j = 0; j + 1 < cl; ++j) {
      if (!whole && !s.drop[j]) continue;
      const int a = cy[j], b = cy[j + 1];
      const int e = s.find(a, b);
      if (e < 0) continue;
      const int m = s.mul[e];
      if (m == 1) {
        s.rx[s.rid[e]] = -1;
      } else {
        const int lo = min(a, b), hi = max(a, b);
        for (int r = first; r < s.nrows; ++r)
          if (s.rx[r] == lo && s.ry[r] == hi) s.rx[r] = -1;
      }
      s.nlive -= m;
      s.cnt[a] -= m;
      s.cnt[b] -= m;
      const int back = s.find(b, a);
      s.unlink(a, e);
      s.unlink(b, back);
    }
    const int adds = add_b >= 0 ? 1 : (star ? nb : 0);
    if (s.nrows + adds > row_cap) {  // squeeze out the dead rows, keeping the order of the live ones
      int w = 0;
      for (int r = 0; r < s.nrows; ++r) {
        const int x = s.rx[r], y = s.ry[r];
        if (x >= 0) { s.rx[w] = x; s.ry[w++] = y; }
      }
      s.nrows = w;
      first = 0;
      for (int v = 0; v < nv; ++v)
        for (int e = s.head[v]; e >= 0; e = s.nxt[e]) s.rid[e] = -1;
      for (int r = 0; r < s.nrows; ++r) {
        const int x = s.rx[r], y = s.ry[r];
        const int f = s.find(x, y);
        if (f >= 0 && s.rid[f] < 0) {  // (a row whose pair lost its entry has none)
          s.rid[f] = r;
          s.rid[s.find(y, x)] = r;
        }
      }
    }
    if (s.nrows + adds > row_cap) { fail(2); break; }  // live rows outgrew the input's count
    app0 = s.nrows;
    if (add_b >= 0) s.add_row(add_a, add_b);
    if (star)
      for (int i = 0; i < nb; ++i) {
        const int x = s.branch[i];
        if (x != hub) s.add_row(x, hub);
      }
    app1 = s.nrows;
  }
  wave_sync();
  int live = 0;
  for (int r = lane; r < s.nrows; r += 64) live += s.rx[r] >= 0;
  int w = wave_total(live);
  if (w > E) {  // more live rows than the component had (rows repeated in both orientations)
    fail(2);
    w = 0;
  }
  int done = 0;
  for (int r0 = 0; r0 < s.nrows && done < w; r0 += 64) {
    const int r = r0 + lane;
    const bool on = r < s.nrows && s.rx[r] >= 0;
    const unsigned long long m = __builtin_amdgcn_ballot_w64(on);
    if (on) rows_out[done + __popcll(m & ((1ULL << lane) - 1ULL))] = make_int2(s.rx[r], s.ry[r]);
    done += __popcll(m);
  }
  if (lane == 0) *ne_out = w;
}

extern __shared__ int post_lds[];

// Block b: component list[b], its state in LDS.
__global__ void __launch_bounds__(64) loops_small(const int *list, const long long *vs, const long long *es, const int2 *rows_in,
                                                  const int *vlist, const float *vertices, const float *radii, int2 *rows_out,
                                                  int *ne_out, int *failed) {
  const int c = list[blockIdx.x];
  const long long v0 = vs[c], e0 = es[c];
  const int nv = int(vs[c + 1] - v0), E = int(es[c + 1] - e0);
  auto s = loop_state<InLds<short> *, InLds<unsigned char> *>((InLds<short> *)post_lds, nv, E);
  loop_lists(s, (InLds<int> *)post_lds, nv, E, rows_in + e0);
  loops_component(s, nv, E, vlist + v0, vertices, radii, rows_out + e0, ne_out + c, failed);
}

// Block b: component list[b], its state at slot starts[b] (ints) of `arena`.
__global__ void __launch_bounds__(64) loops_large(const int *list, const long long *starts, int *arena, const long long *vs,
                                                  const long long *es, const int2 *rows_in, const int *vlist,
                                                  const float *vertices, const float *radii, int2 *rows_out, int *ne_out,
                                                  int *failed) {
  const int c = list[blockIdx.x];
  const long long v0 = vs[c], e0 = es[c];
  const int nv = int(vs[c + 1] - v0), E = int(es[c + 1] - e0);
  InGlobal<int> *at = (InGlobal<int> *)(arena + starts[blockIdx.x]);
  auto s = loop_state<InGlobal<int> *, InGlobal<unsigned char> *>(at, nv, E);
  loop_lists(s, at, nv, E, rows_in + e0);
  loops_component(s, nv, E, vlist + v0, vertices, radii, rows_out + e0, ne_out + c, failed);
}

__global__ void loop_keys_untouched(const int2 *e, const int *root, const int *slot, int m, unsigned long long *keys) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= m) return;
  const int2 x = e[i];
  keys[i] = slot[root[x.x]] < 0 && x.x != x.y
                ? ((unsigned long long)min(x.x, x.y) << 32) | (unsigned long long)max(x.x, x.y)
                : kNone;
}

__global__ void loop_keys_kept(const int2 *rows, const int *ne_out, const long long *es, const long long *vs, const int *vlist,
                               const int *elist, const int *comp_of_edge, int count_edges, unsigned long long *keys) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j >= count_edges) return;
  const int c = comp_of_edge[j];
  if (j - es[c] >= ne_out[c]) return;
  const unsigned a = unsigned(vlist[vs[c] + rows[j].x]), b = unsigned(vlist[vs[c] + rows[j].y]);
  if (a != b) keys[elist[j]] = ((unsigned long long)min(a, b) << 32) | (unsigned long long)max(a, b);
}

__global__ void keep_unemptied(const int *root, const int *slot, const int *ne_out, int n, int *keep) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const int c = slot[root[i]];
  keep[i] = c < 0 || ne_out[c] > 0;
}

DevicePacked remove_loops(Context &ctx, DevicePacked p) {
  if (!p.n() || !p.m()) return p;
  Graph g = build_graph(ctx, p);
  Pieces pc = pieces_of(ctx, g, false);
  if (!pc.count) return p;
  auto s = ctx.stream();
  const long long A = pc.count, M = pc.ne;
  Buffer<int2> rows_out(ctx, size_t(std::max<long long>(M, 1)));
  Buffer<int> ne_out(ctx, A), failed(ctx, 1);
  failed.clear(ctx);
  const Split sp = split_pieces(ctx, pc, [](size_t, size_t nv, size_t E) { return loop_bytes<short>(nv, E); });
  if (sp.nsmall) {
    BROOK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(loops_small), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(kLdsPiece)));
    loops_small<<<unsigned(sp.nsmall), 64, sp.lds, s>>>(sp.small.data(), pc.vs.data(), pc.es.data(), pc.rows.data(),
                                                       pc.vlist.data(), p.vertices.data(), p.radii.data(), rows_out.data(),
                                                       ne_out.data(), failed.data());
    BROOK_LAUNCHED();
  }
  Buffer<int> arena;
  Buffer<long long> starts_dev;
  if (sp.nlarge) {
    std::vector<int> large = sp.large.download(ctx);
    std::vector<long long> starts;
    long long ints = 0;
    for (int c : large) {
      starts.push_back(ints);
      ints += (long long)((loop_bytes<int>(size_t(pc.vs_host[size_t(c) + 1] - pc.vs_host[size_t(c)]),
                                           size_t(pc.es_host[size_t(c) + 1] - pc.es_host[size_t(c)])) + 3) / 4);
    }
    arena = Buffer<int>(ctx, size_t(ints));
    starts_dev = Buffer<long long>(ctx, starts.size());
    starts_dev.upload(ctx, starts.data(), starts.size());
    loops_large<<<unsigned(sp.nlarge), 64, 0, s>>>(sp.large.data(), starts_dev.data(), arena.data(), pc.vs.data(), pc.es.data(),
                                                  pc.rows.data(), pc.vlist.data(), p.vertices.data(), p.radii.data(),
                                                  rows_out.data(), ne_out.data(), failed.data());
    BROOK_LAUNCHED();
  }
  const int failure = read_one(ctx, failed.data());
  if (failure & 1) throw std::runtime_error("remove_loops did not converge");
  if (failure & 2) throw std::runtime_error("remove_loops row capacity exceeded (rows repeated in both orientations)");
  Buffer<unsigned long long> keys(ctx, size_t(std::max(g.m, 1)));
  loop_keys_untouched<<<grid(g.m), kThreads, 0, s>>>(g.e.data(), g.root.data(), pc.slot.data(), g.m, keys.data());
  if (M)
    loop_keys_kept<<<grid(M), kThreads, 0, s>>>(rows_out.data(), ne_out.data(), pc.es.data(), pc.vs.data(), pc.vlist.data(),
                                                pc.elist.data(), pc.comp_of_edge.data(), int(M), keys.data());
  BROOK_LAUNCHED();
  const std::vector<int> kept = ne_out.download(ctx);
  DevicePacked out = edges_from_keys(ctx, std::move(p), g, keys, g.m);
  if (std::find(kept.begin(), kept.end(), 0) == kept.end()) return out;
  Buffer<int> keep(ctx, g.n);
  keep_unemptied<<<grid(g.n), kThreads, 0, s>>>(g.root.data(), pc.slot.data(), ne_out.data(), g.n, keep.data());
  BROOK_LAUNCHED();
  Graph next = build_graph(ctx, out, false);
  return select_vertices(ctx, out, keep, next);
}

// ---------------------------------------------------------------------------------------------
// remove_ticks: one wave per tree with a branch point (post_kernels.cuh:309-405)

// CSR neighbours of the pieces' vertices: a node's rows that start at it, then those that end at
// it, each in row order (a stable sort of both directions by source).
__global__ void csr_entries(const int2 *rows, const long long *vs, const long long *es, const int *comp_of_edge, int M,
                            unsigned *source, unsigned long long *value) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j >= M) return;
  const int c = comp_of_edge[j];
  const unsigned r = unsigned(j - es[c]);
  const int2 x = rows[j];
  source[j] = unsigned(vs[c] + x.x);
  value[j] = ((unsigned long long)unsigned(x.y) << 32) | r;
  source[M + j] = unsigned(vs[c] + x.y);
  value[M + j] = ((unsigned long long)unsigned(x.x) << 32) | r;
}

// off[v]: the first entry whose source is at or past v.
__global__ void csr_offsets(const unsigned *source_sorted, long long total, long long n, long long *off) {
  const long long v = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (v > n) return;
  long long lo = 0, hi = total;
  while (lo < hi) {
    const long long mid = (lo + hi) >> 1;
    if ((long long)source_sorted[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  off[v] = lo;
}

// A binary heap keyed (length, lower end, higher end).
template <class I, class D> struct Heap {
  D len;
  I lo, hi, id, ver;
  int n = 0;
  __device__ bool less(int i, int j) const {
    const double a = len[i], b = len[j];
    return a < b || (a == b && (lo[i] < lo[j] || (lo[i] == lo[j] && hi[i] < hi[j])));
  }
  __device__ void swap(int i, int j) {
    const double l = len[i]; len[i] = len[j]; len[j] = l;
    int t = lo[i]; lo[i] = lo[j]; lo[j] = t;
    t = hi[i]; hi[i] = hi[j]; hi[j] = t;
    t = id[i]; id[i] = id[j]; id[j] = t;
    t = ver[i]; ver[i] = ver[j]; ver[j] = t;
  }
  __device__ void push(double l, int a, int b, int s, int v) {
    int i = n++;
    len[i] = l; lo[i] = min(a, b); hi[i] = max(a, b); id[i] = s; ver[i] = v;
    while (i > 0) {
      const int up = (i - 1) >> 1;
      if (!less(i, up)) break;
      swap(i, up);
      i = up;
    }
  }
  __device__ void pop() {
    if (--n <= 0) return;
    swap(0, n);
    int i = 0;
    for (;;) {
      const int l = 2 * i + 1, r = l + 1;
      int m = i;
      if (l < n && less(l, m)) m = l;
      if (r < n && less(r, m)) m = r;
      if (m == i) break;
      swap(i, m);
      i = m;
    }
  }
};

// A tree's state: I indexes (pointer to short in LDS, int in device memory), D doubles, F floats, B
// bytes. A tree of `critical` vertices of degree 1 or at least 3 has critical - 1 chains between them, at
// most 2 of them ever enter the heap per chain (one at first, one per fusion), and its search stack
// holds roots of subtrees not entered yet, each with a leaf of its own.
template <class I, class D, class F, class B> struct TickState {
  D len;                                   // chains
  Heap<I, D> heap;                         // 2 per chain
  F pos, sdist;                            // 3 nv; stack
  I off, child, row;                       // nv + 1; 2 E: the neighbours
  I bc, slot_head;                         // nv
  I node, parent, root, chain;             // stack
  I su, sv, ver, cf, cla, cn;              // chains
  I snext, sowner;                         // 2 per chain
  I chain_of;                              // E: row -> chain
  B alive, eligible, dead;                 // chains
};
template <class T> size_t tick_bytes(size_t nv, size_t E, size_t critical) {
  const size_t C = critical + 1, H = 2 * C + 2, S = critical + 2;
  return 8 * (C + H) + 4 * (3 * nv + S) + sizeof(T) * (4 * H + nv + 1 + 4 * E + 2 * nv + 4 * S + 6 * C + 4 * C + E) + 3 * C;
}
template <class I, class D, class F, class B> __device__ TickState<I, D, F, B> tick_state(D at, int nv, int E, int critical) {
  const int C = critical + 1, H = 2 * C + 2, S = critical + 2;
  TickState<I, D, F, B> s;
  s.len = at;
  s.heap.len = at + C;
  F f = (F)(at + C + H);
  s.pos = f;
  s.sdist = f + 3 * nv;
  I i = (I)(f + 3 * nv + S);
  auto take = [&](int n) { I p = i; i += n; return p; };
  s.heap.lo = take(H);
  s.heap.hi = take(H);
  s.heap.id = take(H);
  s.heap.ver = take(H);
  s.off = take(nv + 1);
  s.child = take(2 * E);
  s.row = take(2 * E);
  s.bc = take(nv);
  s.slot_head = take(nv);
  s.node = take(S);
  s.parent = take(S);
  s.root = take(S);
  s.chain = take(S);
  s.su = take(C);
  s.sv = take(C);
  s.ver = take(C);
  s.cf = take(C);
  s.cla = take(C);
  s.cn = take(C);
  s.snext = take(2 * C);
  s.sowner = take(2 * C);
  s.chain_of = take(E);
  s.alive = (B)i;
  s.eligible = s.alive + C;
  s.dead = s.eligible + C;
  return s;
}

// keep_rows[r]: row r of the tree stays. off, csr: the CSR from the tree's first vertex on.
template <class I, class D, class F, class B>
__device__ void ticks_component(TickState<I, D, F, B> &s, int nv, int E, const int *vl, const float *vertices, const long long *off,
                                const unsigned long long *csr, double threshold, unsigned char *keep_rows) {
  const int lane = threadIdx.x;
  const long long base = off[0];
  for (int v = lane; v <= nv; v += 64) s.off[v] = int(off[v] - base);
  for (int q = lane; q < 2 * E; q += 64) {
    const unsigned long long x = csr[base + q];
    s.child[q] = int(x >> 32);
    s.row[q] = int(unsigned(x));
  }
  for (int j = lane; j < 3 * nv; j += 64) s.pos[j] = vertices[3LL * vl[j / 3] + j % 3];
  wave_sync();
  auto deg = [&](int v) { return int(s.off[v + 1]) - int(s.off[v]); };
  int start = INT_MAX;
  for (int v = lane; v < nv; v += 64) {
    const int d = deg(v);
    s.bc[v] = d >= 3 ? d : 0;
    s.slot_head[v] = -1;
    if (d == 1) start = min(start, v);
  }
  for (int o = 32; o > 0; o >>= 1) start = min(start, __shfl_xor(start, o, 64));
  wave_sync();
  if (start == INT_MAX) {
    for (int r = lane; r < E; r += 64) keep_rows[r] = 1;
    return;
  }
  int chains = 0, sp = 0;
  s.node[sp] = start;
  s.parent[sp] = -1;
  s.root[sp] = start;
  s.chain[sp] = -1;
  s.sdist[sp++] = 0.0f;
  while (sp) {
    --sp;
    const int node = s.node[sp], parent = s.parent[sp];
    int root = s.root[sp], chain = s.chain[sp];
    float dist = s.sdist[sp];
    const int q0 = s.off[node], q1 = s.off[node + 1], d = q1 - q0;
    if ((d == 1 || d >= 3) && node != root) {  // a chain reaches a critical node: a super-edge
      s.su[chain] = root;
      s.sv[chain] = node;
      s.len[chain] = double(dist);
      s.ver[chain] = 0;
      s.alive[chain] = 1;
      const bool el = deg(root) == 1 || d == 1;
      s.eligible[chain] = el;
      s.snext[2 * chain] = s.slot_head[root];
      s.slot_head[root] = 2 * chain;
      s.snext[2 * chain + 1] = s.slot_head[node];
      s.slot_head[node] = 2 * chain + 1;
      s.sowner[2 * chain] = s.sowner[2 * chain + 1] = chain;
      if (el) s.heap.push(double(dist), root, node, chain, 0);
      dist = 0.0f;
      root = node;
    }
    const float nx = s.pos[3 * node], ny = s.pos[3 * node + 1], nz = s.pos[3 * node + 2];
    for (int q = q0; q < q1; ++q) {
      const int child = s.child[q], row = s.row[q];
      if (child == parent) continue;
      float dx = nx - s.pos[3 * child], dy = ny - s.pos[3 * child + 1], dz = nz - s.pos[3 * child + 2];
      dx *= dx;
      dy *= dy;
      dz *= dz;
      int ch = chain;
      if (node == root) {  // a chain leaves a critical node
        ch = chains++;
        s.cf[ch] = s.cla[ch] = ch;
        s.cn[ch] = -1;
        s.dead[ch] = 0;
        s.alive[ch] = 0;
        s.eligible[ch] = 0;
      }
      s.chain_of[row] = ch;
      s.node[sp] = child;
      s.parent[sp] = node;
      s.root[sp] = root;
      s.chain[sp] = ch;
      s.sdist[sp++] = dist + sqrtf((dx + dy) + dz);
    }
  }
  int nalive = 0;
  for (int k = 0; k < chains; ++k) nalive += s.alive[k];
  while (nalive > 1) {
    while (s.heap.n > 0 && (!s.alive[s.heap.id[0]] || s.ver[s.heap.id[0]] != s.heap.ver[0])) s.heap.pop();
    if (s.heap.n == 0) break;
    const int best = s.heap.id[0];
    const int e1 = s.su[best], e2 = s.sv[best];
    if (s.bc[e1] == 1 && s.bc[e2] == 1) break;
    if (s.len[best] >= threshold) break;
    s.heap.pop();
    for (int k = s.cf[best]; k >= 0; k = s.cn[k]) s.dead[k] = 1;
    s.alive[best] = 0;
    nalive--;
    s.bc[e1] -= 1;
    s.bc[e2] -= 1;
    for (int t = 0; t < 2; ++t) {
      const int v = t ? e2 : e1;
      if (s.bc[v] != 2) continue;
      int a = -1, b = -1;
      for (int k = s.slot_head[v]; k >= 0; k = s.snext[k]) {
        const int o = s.sowner[k];
        if (!s.alive[o] || (s.su[o] != v && s.sv[o] != v) || o == a) continue;
        if (a < 0) a = o;
        else { b = o; break; }
      }
      if (a < 0 || b < 0) { s.bc[v] = 0; continue; }
      const int ea = s.su[a] == v ? s.sv[a] : s.su[a], eb = s.su[b] == v ? s.sv[b] : s.su[b];
      const double la = (0.0 + s.len[a]) + s.len[b];
      s.len[a] = la;
      s.su[a] = ea;
      s.sv[a] = eb;
      s.eligible[a] = 1;
      s.cn[s.cla[a]] = s.cf[b];
      s.cla[a] = s.cla[b];
      s.alive[b] = 0;
      nalive--;
      for (int k = s.slot_head[eb]; k >= 0; k = s.snext[k])
        if (s.sowner[k] == b) s.sowner[k] = a;
      const int ver = s.ver[a] + 1;
      s.ver[a] = ver;
      s.heap.push(la, ea, eb, a, ver);
      s.bc[v] = 0;
    }
  }
  wave_sync();
  for (int r = lane; r < E; r += 64) keep_rows[r] = !s.dead[s.chain_of[r]];
}

// Block b: tree list[b], its state in LDS.
__global__ void __launch_bounds__(64) ticks_small(const int *list, const long long *vs, const long long *es, const int *critical,
                                                  const int *vlist, const float *vertices, const long long *csr_off,
                                                  const unsigned long long *csr, double threshold, unsigned char *keep_rows) {
  const int c = list[blockIdx.x];
  const long long v0 = vs[c], e0 = es[c];
  const int nv = int(vs[c + 1] - v0), E = int(es[c + 1] - e0);
  auto s = tick_state<InLds<short> *, InLds<double> *, InLds<float> *, InLds<unsigned char> *>((InLds<double> *)post_lds, nv, E,
                                                                                             critical[c]);
  ticks_component(s, nv, E, vlist + v0, vertices, csr_off + v0, csr, threshold, keep_rows + e0);
}

// Block b: tree list[b], its state at slot starts[b] (doubles) of `arena`.
__global__ void __launch_bounds__(64) ticks_large(const int *list, const long long *starts, double *arena, const long long *vs,
                                                  const long long *es, const int *critical, const int *vlist,
                                                  const float *vertices, const long long *csr_off,
                                                  const unsigned long long *csr, double threshold, unsigned char *keep_rows) {
  const int c = list[blockIdx.x];
  const long long v0 = vs[c], e0 = es[c];
  const int nv = int(vs[c + 1] - v0), E = int(es[c + 1] - e0);
  auto s = tick_state<InGlobal<int> *, InGlobal<double> *, InGlobal<float> *, InGlobal<unsigned char> *>(
      (InGlobal<double> *)(arena + starts[blockIdx.x]), nv, E, critical[c]);
  ticks_component(s, nv, E, vlist + v0, vertices, csr_off + v0, csr, threshold, keep_rows + e0);
}

__global__ void tick_keep(const int *elist, const unsigned char *keep_rows, int M, int *keep) {
  const int j = blockIdx.x * kThreads + threadIdx.x;
  if (j < M) keep[elist[j]] = keep_rows[j];
}

__global__ void fill_ones(int *out, int n) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = 1;
}

DevicePacked remove_ticks(Context &ctx, DevicePacked p, double threshold) {
  if (threshold == 0 || !p.n() || !p.m()) return p;
  Graph g = build_graph(ctx, p);
  Pieces pc = pieces_of(ctx, g, true);
  if (!pc.count) return p;
  auto s = ctx.stream();
  const long long A = pc.count, N = pc.nv, M = pc.ne;
  if (M > INT32_MAX / 2) throw std::invalid_argument("tick adjacency exceeds int32 capacity");
  Buffer<unsigned> source(ctx, size_t(2 * M)), source_sorted(ctx, size_t(2 * M));
  Buffer<unsigned long long> value(ctx, size_t(2 * M)), csr(ctx, size_t(2 * M));
  csr_entries<<<grid(M), kThreads, 0, s>>>(pc.rows.data(), pc.vs.data(), pc.es.data(), pc.comp_of_edge.data(), int(M),
                                           source.data(), value.data());
  BROOK_LAUNCHED();
  Buffer<unsigned char> scratch;
  with_scratch(ctx, scratch, [&](void *t, size_t &b) {
    return hipcub::DeviceRadixSort::SortPairs(t, b, source.data(), source_sorted.data(), value.data(), csr.data(), int(2 * M), 0,
                                              bits_for(N), s);
  });
  Buffer<long long> off(ctx, size_t(N) + 1);
  csr_offsets<<<grid(N + 1), kThreads, 0, s>>>(source_sorted.data(), 2 * M, N, off.data());
  BROOK_LAUNCHED();
  Buffer<unsigned char> keep_rows(ctx, size_t(M));
  Buffer<int> critical(ctx, size_t(A));
  critical.upload(ctx, pc.critical.data(), size_t(A));
  const Split sp = split_pieces(ctx, pc, [&](size_t c, size_t nv, size_t E) { return tick_bytes<short>(nv, E, size_t(pc.critical[c])); });
  if (sp.nsmall) {
    BROOK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(ticks_small), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(kLdsPiece)));
    ticks_small<<<unsigned(sp.nsmall), 64, sp.lds, s>>>(sp.small.data(), pc.vs.data(), pc.es.data(), critical.data(),
                                                       pc.vlist.data(), p.vertices.data(), off.data(), csr.data(), threshold,
                                                       keep_rows.data());
    BROOK_LAUNCHED();
  }
  Buffer<double> arena;
  Buffer<long long> starts_dev;
  if (sp.nlarge) {
    std::vector<int> large = sp.large.download(ctx);
    std::vector<long long> starts;
    long long doubles = 0;
    for (int c : large) {
      starts.push_back(doubles);
      doubles += (long long)((tick_bytes<int>(size_t(pc.vs_host[size_t(c) + 1] - pc.vs_host[size_t(c)]),
                                              size_t(pc.es_host[size_t(c) + 1] - pc.es_host[size_t(c)]),
                                              size_t(pc.critical[size_t(c)])) + 7) / 8);
    }
    arena = Buffer<double>(ctx, size_t(doubles));
    starts_dev = Buffer<long long>(ctx, starts.size());
    starts_dev.upload(ctx, starts.data(), starts.size());
    ticks_large<<<unsigned(sp.nlarge), 64, 0, s>>>(sp.large.data(), starts_dev.data(), arena.data(), pc.vs.data(), pc.es.data(),
                                                  critical.data(), pc.vlist.data(), p.vertices.data(), off.data(), csr.data(),
                                                  threshold, keep_rows.data());
    BROOK_LAUNCHED();
  }
  Buffer<int> keep(ctx, size_t(g.m));
  fill_ones<<<grid(g.m), kThreads, 0, s>>>(keep.data(), g.m);
  tick_keep<<<grid(M), kThreads, 0, s>>>(pc.elist.data(), keep_rows.data(), int(M), keep.data());
  BROOK_LAUNCHED();
  return select_edges(ctx, std::move(p), keep, g);
}

// ---------------------------------------------------------------------------------------------
// join_components (post.cu:521-648, post_kernels.cuh:210-306)

__global__ void join_statistics(const int *root, const int *vlabel, const float *radii, int n, int *ncomp, unsigned *rmax) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int l = i < n ? vlabel[i] : -1;
  if (i < n && root[i] == i) atomicAdd(ncomp + l, 1);
  const float r = i < n ? radii[i] : 0.0f;
  unsigned top = r > 0 ? __float_as_uint(r) : 0u;
  // vertices come label by label: a wave of one label sends one maximum
  const int first = __shfl(l, 0, 64);
  if (__all(l == first)) {
    for (int o = 32; o > 0; o >>= 1) top = max(top, unsigned(__shfl_xor(int(top), o, 64)));
    if ((threadIdx.x & 63) != 0) top = 0u;
  }
  if (top && l >= 0) atomicMax(rmax + l, top);
}

// Cell of a vertex of a label with several components: (rank, floor(coordinate / bound)); the others'
// rank is LLONG_MAX. range: least and greatest rank, x, y, z over the members (LLONG_MAX, LLONG_MIN
// before).
__global__ void join_cells(const int *vlabel, const int *rank, const double *bound, const float *v, int n, long long *kl,
                           long long *kx, long long *ky, long long *kz, int *index, long long *range) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  const int r = i < n ? rank[vlabel[i]] : -1;
  long long k[3] = {0, 0, 0};
  if (r >= 0) {
    const double b = bound[r];
    for (int a = 0; a < 3; ++a) k[a] = (long long)floor(double(v[3LL * i + a]) / b);
  }
  if (i < n) {
    index[i] = i;
    kl[i] = r < 0 ? LLONG_MAX : r;
    kx[i] = k[0];
    ky[i] = k[1];
    kz[i] = k[2];
  }
  for (int a = 0; a < 3; ++a) {
    long long lo = r < 0 ? LLONG_MAX : k[a], hi = r < 0 ? LLONG_MIN : k[a];
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o, 64));
      hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if ((threadIdx.x & 63) == 0 && lo <= hi) {
      atomicMin(range + 2 * a, lo);
      atomicMax(range + 2 * a + 1, hi);
    }
  }
}

__global__ void permute_key(const long long *key, const int *order, int n, long long *out) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = key[order[i]];
}

__global__ void iota(int *out, int n) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = i;
}

// A vertex in cell order: what its neighbours' searches read.
struct alignas(16) CellVertex {
  float x, y, z;
  int root;
};
__global__ void cell_vertices(const int *order, const float *v, const int *root, int n, CellVertex *out) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p >= n) return;
  const int i = order[p];
  out[p] = CellVertex{v[3LL * i], v[3LL * i + 1], v[3LL * i + 2], root[i]};
}

// Cells whose four coordinates fit one 64-bit key (z in the low bits): the sorted keys.
struct CellRange {
  long long least[3];
  int bits[3];
  unsigned long long most[3];  // greatest coordinate, from the least
};
__global__ void pack_cells(const long long *kl, const long long *kx, const long long *ky, const long long *kz, int n, CellRange r,
                           unsigned long long *key) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  if (kl[i] == LLONG_MAX) { key[i] = kNone; return; }
  const unsigned long long x = (unsigned long long)(kx[i] - r.least[0]), y = (unsigned long long)(ky[i] - r.least[1]),
                           z = (unsigned long long)(kz[i] - r.least[2]);
  key[i] = ((((unsigned long long)kl[i] << r.bits[0] | x) << r.bits[1]) | y) << r.bits[2] | z;
}
struct PackedCells {
  const unsigned long long *key;  // per position
  int n;
  CellRange r;
  struct Cell { unsigned long long key; };
  __device__ Cell at(int pos) const { return Cell{key[pos]}; }
  __device__ static Cell from_lane(const Cell &c, int lane) { return Cell{__shfl(c.key, lane, 64)}; }
  __device__ static bool same(const Cell &a, const Cell &b) { return a.key == b.key; }
  __device__ bool member(const Cell &c) const { return c.key != kNone; }
  __device__ int rank(const Cell &c) const { return int(c.key >> (r.bits[0] + r.bits[1] + r.bits[2])); }
  // The key of cell (x + dx, y + dy, z - 1) (end false) or (x + dx, y + dy, z + 1); false: no such column.
  __device__ bool column(const Cell &c, int dx, int dy, bool end, unsigned long long &k) const {
    auto field = [&](int shift, int bits) { return (c.key >> shift) & ((1ULL << bits) - 1ULL); };
    const unsigned long long x = field(r.bits[1] + r.bits[2], r.bits[0]), y = field(r.bits[2], r.bits[1]), z = field(0, r.bits[2]);
    if ((dx < 0 && x == 0) || (dx > 0 && x == r.most[0]) || (dy < 0 && y == 0) || (dy > 0 && y == r.most[1])) return false;
    const unsigned long long nz = end ? (z < r.most[2] ? z + 1 : z) : (z > 0 ? z - 1 : z);
    k = c.key >> (r.bits[0] + r.bits[1] + r.bits[2]);
    k = ((((k << r.bits[0]) | (x + dx)) << r.bits[1]) | (y + dy)) << r.bits[2] | nz;
    return true;
  }
  // First position at or past the column's first cell, or past its last; whether `pos` is past it.
  __device__ int bound(const Cell &c, int dx, int dy, bool end) const {
    unsigned long long k;
    if (!column(c, dx, dy, end, k)) return 0;
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (key[mid] < k || (end && key[mid] == k)) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  }
  __device__ bool past(int pos, const Cell &c, int dx, int dy) const {
    unsigned long long k;
    return pos >= n || !column(c, dx, dy, true, k) || key[pos] > k;
  }
};

// Cells of any coordinates (a label whose radii are all 0 has cells of a millionth): four keys per vertex.
struct WideCells {
  const int *order;  // position -> vertex
  const long long *kl, *kx, *ky, *kz;  // per vertex
  int n;
  struct Cell { long long l, x, y, z; };
  __device__ Cell at(int pos) const { const int v = order[pos]; return Cell{kl[v], kx[v], ky[v], kz[v]}; }
  __device__ static Cell from_lane(const Cell &c, int lane) {
    return Cell{__shfl(c.l, lane, 64), __shfl(c.x, lane, 64), __shfl(c.y, lane, 64), __shfl(c.z, lane, 64)};
  }
  __device__ static bool same(const Cell &a, const Cell &b) { return a.l == b.l && a.x == b.x && a.y == b.y && a.z == b.z; }
  __device__ bool member(const Cell &c) const { return c.l != LLONG_MAX; }
  __device__ int rank(const Cell &c) const { return int(c.l); }
  __device__ int cmp(int pos, const Cell &c) const {
    const int v = order[pos];
    if (kl[v] != c.l) return kl[v] < c.l ? -1 : 1;
    if (kx[v] != c.x) return kx[v] < c.x ? -1 : 1;
    if (ky[v] != c.y) return ky[v] < c.y ? -1 : 1;
    if (kz[v] != c.z) return kz[v] < c.z ? -1 : 1;
    return 0;
  }
  __device__ bool column(const Cell &c, int dx, int dy, bool end, Cell &k) const {
    if (c.x == (dx < 0 ? LLONG_MIN : LLONG_MAX) && dx) return false;
    if (c.y == (dy < 0 ? LLONG_MIN : LLONG_MAX) && dy) return false;
    k = Cell{c.l, c.x + dx, c.y + dy, end ? (c.z < LLONG_MAX ? c.z + 1 : c.z) : (c.z > LLONG_MIN ? c.z - 1 : c.z)};
    return true;
  }
  __device__ int bound(const Cell &c, int dx, int dy, bool end) const {
    Cell k;
    if (!column(c, dx, dy, end, k)) return 0;
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1, o = cmp(mid, k);
      if (o < 0 || (end && o == 0)) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  }
  __device__ bool past(int pos, const Cell &c, int dx, int dy) const {
    Cell k;
    return pos >= n || !column(c, dx, dy, true, k) || cmp(pos, k) > 0;
  }
};

constexpr int kJoinTable = 16, kFewCells = 16;

// Per vertex of a joinable label: for each component above its own within reach, the nearest vertex
// (ties by the lower index); a vertex meeting more components than its table holds sends the excess
// straight out. Candidates go to the places *count gives out, in no order (they are sorted by all
// their fields), none at or past `cap` (*count then says how many there are).
// A thread per vertex in cell order, so that a wave's vertices lie in one or a few cells: per cell, lanes
// find the bounds of its 9 columns of three cells (contiguous positions), then the cell's lanes
// walk the same positions together, from one array in that order. (166 k vertices of 150 skeletons:
// 0.33 ms; a search of 27 cells per vertex through the sort order, once to count and once to write,
// took 2.3 ms.) Where a wave's vertices lie in more than kFewCells cells, that is a search after another for
// a lane or two each, and every lane searches the columns of its own cell instead: 200 k vertices without
// radii, a cell each, 1.80 ms for the whole step, a cell at a time 2.19 (27 cells per vertex 1.70); radii of a
// tenth of the spacing 1.86, 2.04 (2.51). Limits of 8, 16 and 32 cells are within 3 % of each other.
template <class Cells>
__global__ void __launch_bounds__(kThreads) join_candidates(Cells cells, const CellVertex *cv, const int *order,
                                                           const double *bound, unsigned long long *count, unsigned long long cap,
                                                           int *oa, int *ob,
                                                           double *od, int *ov, int *ou) {
  const int p = blockIdx.x * kThreads + threadIdx.x, lane = int(threadIdx.x) & 63;
  const int at = p < cells.n ? p : cells.n - 1;
  const typename Cells::Cell mine = cells.at(at);
  const CellVertex me = cv[at];
  const int i = order[at];
  int tb[kJoinTable], tu[kJoinTable];
  double td[kJoinTable];
  int nt = 0;
  auto emit = [&](int cj, double d, int j) {
    const unsigned long long o = atomicAdd(count, 1ULL);
    if (o >= cap) return;
    oa[o] = me.root;
    ob[o] = cj;
    od[o] = d;
    ov[o] = i;
    ou[o] = j;
  };
  auto look = [&](int q, double bnd, float b32) {
    const CellVertex o = cv[q];
    if (o.root <= me.root) return;
    const float fx = o.x - me.x, fy = o.y - me.y, fz = o.z - me.z;
    if ((fx * fx + fy * fy) + fz * fz > b32) return;
    const double ex = double(o.x) - double(me.x), ey = double(o.y) - double(me.y), ez = double(o.z) - double(me.z);
    const double d = sqrt((ex * ex + ey * ey) + ez * ez);
    if (!(d < bnd)) return;
    const int j = order[q];
    int t = -1;
    for (int k = 0; k < nt; ++k)
      if (tb[k] == o.root) { t = k; break; }
    if (t >= 0) {
      if (d < td[t] || (d == td[t] && j < tu[t])) { td[t] = d; tu[t] = j; }
    } else if (nt < kJoinTable) {
      tb[nt] = o.root; td[nt] = d; tu[nt] = j; nt++;
    } else {
      emit(o.root, d, j);
    }
  };
  auto squared = [](double bnd) {
    const float b = float(bnd);
    return b * b * 1.0001f + 1e-30f;
  };
  const bool member = p < cells.n && cells.member(mine);
  const typename Cells::Cell before = Cells::from_lane(mine, lane ? lane - 1 : 0);
  unsigned long long left = __builtin_amdgcn_ballot_w64(member);
  if (__popcll(__builtin_amdgcn_ballot_w64(member && (lane == 0 || !Cells::same(mine, before)))) > kFewCells) {
    if (member) {
      const double bnd = bound[cells.rank(mine)];
      const float b32 = squared(bnd);
      for (int c = 0; c < 9; ++c) {
        const int dx = c % 3 - 1, dy = c / 3 - 1, q0 = cells.bound(mine, dx, dy, false);
        if (cells.past(q0, mine, dx, dy)) continue;
        const int q1 = cells.bound(mine, dx, dy, true);
        for (int q = q0; q < q1; ++q) look(q, bnd, b32);
      }
    }
    left = 0;
  }
  while (left) {
    const int leader = __ffsll((long long)left) - 1;
    const typename Cells::Cell cell = Cells::from_lane(mine, leader);
    const int col = lane >> 1;  // lanes 2c, 2c + 1: column c's begin and end
    const int b = lane < 18 ? cells.bound(cell, col % 3 - 1, col / 3 - 1, lane & 1) : 0;
    const bool here = ((left >> lane) & 1ULL) && Cells::same(mine, cell);
    left &= ~__builtin_amdgcn_ballot_w64(here);
    const double bnd = bound[cells.rank(cell)];
    const float b32 = squared(bnd);
    for (int c = 0; c < 9; ++c) {
      const int q0 = __shfl(b, 2 * c, 64), q1 = __shfl(b, 2 * c + 1, 64);
      for (int q = q0; q < q1; ++q)
        if (here) look(q, bnd, b32);
    }
  }
  for (int k = 0; k < nt; ++k) emit(tb[k], td[k], tu[k]);
}

__global__ void candidate_key(const int *order, int n, const int *a, const int *b, const double *d, const int *va, const int *vb,
                              int pass, unsigned long long *key) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const int p = order[i];
  if (pass == 0) key[i] = ((unsigned long long)min(va[p], vb[p]) << 32) | (unsigned long long)max(va[p], vb[p]);
  else if (pass == 1) key[i] = (unsigned long long)__double_as_longlong(d[p]);
  else key[i] = ((unsigned long long)unsigned(a[p]) << 32) | (unsigned long long)unsigned(b[p]);
}

__global__ void first_of_pair(const int *order, int n, const int *a, const int *b, int *flag) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  flag[i] = i == 0 || a[order[i]] != a[order[i - 1]] || b[order[i]] != b[order[i - 1]];
}

__global__ void root_flags(const int *root, const int *vlabel, const int *rank, int n, int *flag) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n) flag[i] = root[i] == i && rank[vlabel[i]] >= 0;
}

// A component's position among its label's components (ascending root).
__global__ void root_positions(const int *flag, const int *pos, const int *vlabel, const int *rank, const long long *cs, int n,
                               int *local) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < n && flag[i]) local[i] = int(pos[i] - cs[rank[vlabel[i]]]);
}

__global__ void compact_pairs(const int *order, const int *flag, const int *fpos, int n, const int *a, const int *b,
                              const double *d, const int *va, const int *vb, const int *local, int *cx, int *cy, double *dd,
                              int *pa, int *pb) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n || !flag[i]) return;
  const int p = order[i], j = fpos[i];
  cx[j] = local[a[p]];
  cy[j] = local[b[p]];
  dd[j] = d[p];
  pa[j] = va[p];
  pb[j] = vb[p];
}

// One lane per label: the greedy fusion over the label's candidate list [ps, pe).
__global__ void join_fuse(int labels, const long long *ps, const long long *cs, const double *reach, int *cx, int *cy,
                          const double *dd, const int *va, const int *vb, const float *radii, unsigned char *alive, int *pos,
                          int *slot, int *out_a, int *out_b, int *made) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= labels) return;
  const long long p0 = ps[l], p1 = ps[l + 1], c0 = cs[l];
  const int nc = int(cs[l + 1] - c0);
  int *POS = pos + c0, *SLOT = slot + c0;
  for (int k = 0; k < nc; ++k) { POS[k] = k; SLOT[k] = -1; }
  for (long long q = p0; q < p1; ++q) alive[q] = 1;
  int fusions = 0, count = 0;
  for (;;) {
    long long best = -1;
    float bd = 0.0f;
    int bi = 0, bj = 0;
    for (long long q = p0; q < p1; ++q) {
      if (!alive[q]) continue;
      const double d = dd[q];
      if (d > double(radii[va[q]] + radii[vb[q]])) continue;  // blocked by the radii
      const float d32 = float(d);
      int ia = POS[cx[q]], ib = POS[cy[q]];
      if (ia > ib) { const int t = ia; ia = ib; ib = t; }
      if (best < 0 || d32 < bd || (d32 == bd && (ia < bi || (ia == bi && ib < bj)))) { best = q; bd = d32; bi = ia; bj = ib; }
    }
    if (best < 0 || double(bd) > reach[l]) break;
    const int X = cx[best], Y = cy[best];
    out_a[c0 + count] = va[best];
    out_b[c0 + count] = vb[best];
    count++;
    alive[best] = 0;
    fusions++;
    for (long long q = p0; q < p1; ++q) {  // Y joins X; per other cluster the nearer candidate stays
      if (!alive[q]) continue;
      if (cx[q] == Y) cx[q] = X;
      if (cy[q] == Y) cy[q] = X;
      if (cx[q] == cy[q]) { alive[q] = 0; continue; }
      if (cx[q] != X && cy[q] != X) continue;
      const int k = cx[q] == X ? cy[q] : cx[q];
      if (SLOT[k] < 0) { SLOT[k] = int(q - p0); continue; }
      const long long o = p0 + SLOT[k];
      const int lq = min(va[q], vb[q]), hq = max(va[q], vb[q]), lo = min(va[o], vb[o]), ho = max(va[o], vb[o]);
      const bool q_wins = dd[q] < dd[o] || (dd[q] == dd[o] && (lq < lo || (lq == lo && hq < ho)));
      if (q_wins) { alive[o] = 0; SLOT[k] = int(q - p0); }
      else alive[q] = 0;
    }
    for (long long q = p0; q < p1; ++q)
      if (alive[q]) { SLOT[cx[q]] = -1; SLOT[cy[q]] = -1; }
    POS[X] = -fusions;  // the newest fusion heads the list
  }
  made[l] = count;
}

__global__ void pair_label_offsets(const int *pa, int np, const int *vlabel, const int *rank, int labels, long long *ps) {
  const int l = blockIdx.x * kThreads + threadIdx.x;
  if (l > labels) return;
  int lo = 0, hi = np;  // first candidate whose label rank is >= l
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (rank[vlabel[pa[mid]]] < l) lo = mid + 1;
    else hi = mid;
  }
  ps[l] = lo;
}

__global__ void join_keys(const int2 *e, int m, const int *out_a, const int *out_b, const long long *cs, const int *made,
                          int labels, int roots, unsigned long long *keys) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < m) keys[i] = ((unsigned long long)min(e[i].x, e[i].y) << 32) | (unsigned long long)max(e[i].x, e[i].y);
  if (i < roots) {
    int lo = 0, hi = labels;  // the label whose component range holds i
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (cs[mid] <= i) lo = mid;
      else hi = mid;
    }
    unsigned long long key = kNone;
    if (i - cs[lo] < made[lo])
      key = ((unsigned long long)min(out_a[i], out_b[i]) << 32) | (unsigned long long)max(out_a[i], out_b[i]);
    keys[m + i] = key;
  }
}

DevicePacked join_components(Context &ctx, DevicePacked input) {
  DevicePacked p = prune_unused(ctx, std::move(input));
  if (!p.n() || !p.m()) return p;
  Graph g = build_graph(ctx, p);
  auto s = ctx.stream();
  Buffer<int> ncomp(ctx, g.k);
  Buffer<unsigned> rmax(ctx, g.k);
  ncomp.clear(ctx);
  rmax.clear(ctx);
  join_statistics<<<grid(g.n), kThreads, 0, s>>>(g.root.data(), g.vlabel.data(), p.radii.data(), g.n, ncomp.data(), rmax.data());
  BROOK_LAUNCHED();
  const std::vector<int> nc = ncomp.download(ctx);
  const std::vector<unsigned> bits = rmax.download(ctx);
  std::vector<int> rank(g.k, -1);
  std::vector<double> reach, bound;
  std::vector<long long> cs{0};
  for (int l = 0; l < g.k; ++l)
    if (nc[l] > 1) {
      rank[l] = int(reach.size());
      float r;
      std::memcpy(&r, &bits[l], 4);
      const double x = std::max(2.0 * double(r), 0.0);
      reach.push_back(x);
      bound.push_back(x + 0.000001);
      cs.push_back(cs.back() + nc[l]);
    }
  const int labels = int(reach.size()), roots = int(cs.back());
  if (!labels) return p;
  Buffer<int> rank_dev(ctx, g.k);
  rank_dev.upload(ctx, rank.data(), g.k);
  Buffer<double> reach_dev(ctx, labels), bound_dev(ctx, labels);
  reach_dev.upload(ctx, reach.data(), labels);
  bound_dev.upload(ctx, bound.data(), labels);
  Buffer<long long> cs_dev(ctx, cs.size());
  cs_dev.upload(ctx, cs.data(), cs.size());
  // cells, sorted by (rank, x, y, z): one key where the coordinates' ranges fit 64 bits, else a stable
  // sort per coordinate, least significant first
  Buffer<long long> kl(ctx, g.n), kx(ctx, g.n), ky(ctx, g.n), kz(ctx, g.n), range_dev(ctx, 6);
  Buffer<int> order(ctx, g.n), order_sorted(ctx, g.n);
  long long range[6] = {LLONG_MAX, LLONG_MIN, LLONG_MAX, LLONG_MIN, LLONG_MAX, LLONG_MIN};
  range_dev.upload(ctx, range, 6);
  join_cells<<<grid(g.n), kThreads, 0, s>>>(g.vlabel.data(), rank_dev.data(), bound_dev.data(), p.vertices.data(), g.n, kl.data(),
                                            kx.data(), ky.data(), kz.data(), order.data(), range_dev.data());
  BROOK_LAUNCHED();
  {
    const std::vector<long long> h = range_dev.download(ctx);
    std::copy(h.begin(), h.end(), range);
  }
  CellRange cr{};
  int key_bits = bits_for(labels);
  for (int a = 0; a < 3; ++a) {
    cr.least[a] = range[2 * a];
    cr.most[a] = (unsigned long long)range[2 * a + 1] - (unsigned long long)range[2 * a];
    while (cr.bits[a] < 64 && (cr.most[a] >> cr.bits[a])) ++cr.bits[a];
    key_bits += cr.bits[a];
  }
  const bool packed = key_bits < 64;  // kNone, of the others, sorts last
  Buffer<unsigned char> scratch;
  Buffer<unsigned long long> cell_key(ctx, packed ? size_t(g.n) : 1);
  if (packed) {
    Buffer<unsigned long long> key(ctx, g.n);
    pack_cells<<<grid(g.n), kThreads, 0, s>>>(kl.data(), kx.data(), ky.data(), kz.data(), g.n, cr, key.data());
    BROOK_LAUNCHED();
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortPairs(t, b, key.data(), cell_key.data(), order.data(), order_sorted.data(), g.n, 0,
                                                key_bits + 1, s);
    });
    std::swap(order, order_sorted);
  } else {
    Buffer<long long> key(ctx, g.n), key_sorted(ctx, g.n);
    for (const Buffer<long long> *k : {&kz, &ky, &kx, &kl}) {
      permute_key<<<grid(g.n), kThreads, 0, s>>>(k->data(), order.data(), g.n, key.data());
      BROOK_LAUNCHED();
      with_scratch(ctx, scratch, [&](void *t, size_t &b) {
        return hipcub::DeviceRadixSort::SortPairs(t, b, key.data(), key_sorted.data(), order.data(), order_sorted.data(), g.n, 0, 64, s);
      });
      std::swap(order, order_sorted);
    }
  }
  Buffer<CellVertex> cell_verts(ctx, g.n);
  cell_vertices<<<grid(g.n), kThreads, 0, s>>>(order.data(), p.vertices.data(), g.root.data(), g.n, cell_verts.data());
  BROOK_LAUNCHED();
  Buffer<int> ca, cb, cv, cu;
  Buffer<double> cd;
  Buffer<unsigned long long> found(ctx, 1);
  unsigned long long total = 0;
  for (unsigned long long cap = std::max(g.n, 4096);; cap = total) {
    ca = Buffer<int>(ctx, cap);
    cb = Buffer<int>(ctx, cap);
    cv = Buffer<int>(ctx, cap);
    cu = Buffer<int>(ctx, cap);
    cd = Buffer<double>(ctx, cap);
    found.clear(ctx);
    if (packed)
      join_candidates<<<grid(g.n), kThreads, 0, s>>>(PackedCells{cell_key.data(), g.n, cr}, cell_verts.data(), order.data(),
                                                     bound_dev.data(), found.data(), cap, ca.data(), cb.data(), cd.data(),
                                                     cv.data(), cu.data());
    else
      join_candidates<<<grid(g.n), kThreads, 0, s>>>(WideCells{order.data(), kl.data(), kx.data(), ky.data(), kz.data(), g.n},
                                                     cell_verts.data(), order.data(), bound_dev.data(), found.data(), cap, ca.data(),
                                                     cb.data(), cd.data(), cv.data(), cu.data());
    BROOK_LAUNCHED();
    total = read_one(ctx, found.data());
    if (total > (unsigned long long)INT32_MAX) throw std::invalid_argument("join candidates exceed int32 capacity");
    if (total <= cap) break;
  }
  if (!total) return p;
  const int nt = int(total);
  // candidates by (A, B, distance, lower vertex, higher vertex); the first of each (A, B) stays
  Buffer<int> porder(ctx, nt), porder_sorted(ctx, nt);
  Buffer<unsigned long long> pkey(ctx, nt), pkey_sorted(ctx, nt);
  iota<<<grid(nt), kThreads, 0, s>>>(porder.data(), nt);
  for (int pass = 0; pass < 3; ++pass) {
    candidate_key<<<grid(nt), kThreads, 0, s>>>(porder.data(), nt, ca.data(), cb.data(), cd.data(), cv.data(), cu.data(), pass,
                                                pkey.data());
    BROOK_LAUNCHED();
    with_scratch(ctx, scratch, [&](void *t, size_t &b) {
      return hipcub::DeviceRadixSort::SortPairs(t, b, pkey.data(), pkey_sorted.data(), porder.data(), porder_sorted.data(), nt, 0,
                                                64, s);
    });
    std::swap(porder, porder_sorted);
  }
  Buffer<int> first(ctx, nt + 1), fpos(ctx, nt + 1);
  first_of_pair<<<grid(nt), kThreads, 0, s>>>(porder.data(), nt, ca.data(), cb.data(), first.data());
  BROOK_HIP(hipMemsetAsync(first.data() + nt, 0, 4, s));
  exclusive_sum(ctx, first.data(), fpos.data(), nt + 1);
  const int np = read_one(ctx, fpos.data() + nt);
  Buffer<int> rflag(ctx, g.n + 1), rpos(ctx, g.n + 1), local(ctx, g.n);
  root_flags<<<grid(g.n), kThreads, 0, s>>>(g.root.data(), g.vlabel.data(), rank_dev.data(), g.n, rflag.data());
  BROOK_HIP(hipMemsetAsync(rflag.data() + g.n, 0, 4, s));
  exclusive_sum(ctx, rflag.data(), rpos.data(), g.n + 1);
  root_positions<<<grid(g.n), kThreads, 0, s>>>(rflag.data(), rpos.data(), g.vlabel.data(), rank_dev.data(), cs_dev.data(), g.n,
                                                local.data());
  Buffer<int> px(ctx, np), py(ctx, np), pa(ctx, np), pb(ctx, np);
  Buffer<double> pd(ctx, np);
  compact_pairs<<<grid(nt), kThreads, 0, s>>>(porder.data(), first.data(), fpos.data(), nt, ca.data(), cb.data(), cd.data(), cv.data(),
                                              cu.data(), local.data(), px.data(), py.data(), pd.data(), pa.data(), pb.data());
  Buffer<long long> ps(ctx, size_t(labels) + 1);
  pair_label_offsets<<<grid(labels + 1), kThreads, 0, s>>>(pa.data(), np, g.vlabel.data(), rank_dev.data(), labels, ps.data());
  BROOK_LAUNCHED();
  Buffer<unsigned char> alive(ctx, np);
  Buffer<int> pos(ctx, roots), slot(ctx, roots), out_a(ctx, roots), out_b(ctx, roots), made(ctx, labels);
  join_fuse<<<unsigned((labels + 63) / 64), 64, 0, s>>>(labels, ps.data(), cs_dev.data(), reach_dev.data(), px.data(), py.data(),
                                                       pd.data(), pa.data(), pb.data(), p.radii.data(), alive.data(), pos.data(),
                                                       slot.data(), out_a.data(), out_b.data(), made.data());
  BROOK_LAUNCHED();
  const std::vector<int> mh = made.download(ctx);
  if (*std::max_element(mh.begin(), mh.end()) == 0) return p;  // no join: the edges keep their order
  const int count = g.m + roots;
  Buffer<unsigned long long> keys(ctx, count);
  join_keys<<<grid(std::max(g.m, roots)), kThreads, 0, s>>>(g.e.data(), g.m, out_a.data(), out_b.data(), cs_dev.data(), made.data(),
                                                           labels, roots, keys.data());
  BROOK_LAUNCHED();
  return edges_from_keys(ctx, std::move(p), g, keys, count);
}

}  // namespace

DevicePacked upload_packed(Context &ctx, const PackedView &view) {
  DevicePacked p;
  p.labels.assign(view.labels, view.labels + view.skeletons);
  p.voff.assign(view.v_off, view.v_off + view.skeletons + 1);
  p.eoff.assign(view.e_off, view.e_off + view.skeletons + 1);
  p.anisotropy = view.anisotropy;
  const size_t n = size_t(std::max<int64_t>(p.n(), 0)), m = size_t(std::max<int64_t>(p.m(), 0));
  p.vertices = Buffer<float>(ctx, std::max<size_t>(3 * n, 1));
  p.radii = Buffer<float>(ctx, std::max<size_t>(n, 1));
  p.edges = Buffer<uint32_t>(ctx, std::max<size_t>(2 * m, 1));
  auto s = ctx.stream();
  if (n) {
    BROOK_HIP(hipMemcpyAsync(p.vertices.data(), view.vertices, 12 * n, hipMemcpyDefault, s));
    BROOK_HIP(hipMemcpyAsync(p.radii.data(), view.radii, 4 * n, hipMemcpyDefault, s));
  }
  if (m) BROOK_HIP(hipMemcpyAsync(p.edges.data(), view.edges, 8 * m, hipMemcpyDefault, s));
  ctx.synchronize();
  return p;
}

Packed download_packed(Context &ctx, const DevicePacked &p) {
  Packed out;
  out.labels = p.labels;
  out.v_off.assign(p.voff.begin(), p.voff.end());
  out.e_off.assign(p.eoff.begin(), p.eoff.end());
  out.anisotropy = p.anisotropy;
  out.vertices = p.vertices.download(ctx, size_t(3 * p.n()));
  out.radii = p.radii.download(ctx, size_t(p.n()));
  out.edges = p.edges.download(ctx, size_t(2 * p.m()));
  return out;
}

DevicePacked postprocess(Context &ctx, DevicePacked p, PostStep step, double a, double b) {
  switch (step) {
    case PostStep::dust: return remove_dust(ctx, std::move(p), a);
    case PostStep::loops: return remove_loops(ctx, std::move(p));
    case PostStep::join: return join_components(ctx, std::move(p));
    case PostStep::ticks: return remove_ticks(ctx, std::move(p), a);
    case PostStep::prune: return prune_unused(ctx, std::move(p));
    case PostStep::all: break;
  }
  p = remove_dust(ctx, std::move(p), a);
  p = remove_loops(ctx, std::move(p));
  p = join_components(ctx, std::move(p));
  p = remove_ticks(ctx, std::move(p), b);
  return prune_unused(ctx, std::move(p));
}

std::vector<int64_t> skeleton_components(Context &ctx, const DevicePacked &p) {
  Graph g = build_graph(ctx, p);
  std::vector<int> r = g.root.download(ctx, size_t(g.n));
  return std::vector<int64_t>(r.begin(), r.end());
}

}  // namespace brook
