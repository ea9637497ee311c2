// Multi-label anisotropic Euclidean distance transform on gfx950, with the reference's rounding
// rule (edt_kernels.cuh:15-144, edt.cu:12-23): squared x-distances from a float32 accumulation
// table, y/z lower envelopes with float64 intersections, sqrtf at the end.
//
// Layout for HBM: the x pass gives each row to one wave (64 consecutive voxels per load, run
// boundaries from two ballots, no atomics); the y and z passes take whole lines into LDS, a block a
// stretch of neighbouring ones, and halve for each voxel's nearest vertex. Background runs are never
// evaluated (their values are discarded by the finish rule) and the last pass fuses sqrt, the
// background zero and the per-label maximum.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "stages.hpp"

namespace brook {
namespace {

template <class CC, int MAXCH>
__global__ void __launch_bounds__(256) edt_x(const CC *cc, int sx, int rows, const float *acc, int bb, float *D) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;  // whole wave
  const long long base = (long long)row * sx;
  const int nch = (sx + 63) >> 6;
  CC lab[MAXCH];
  int cst[MAXCH];
  int carry = 0;
  CC tail = CC(0);
#pragma unroll
  for (int j = 0; j < MAXCH; ++j) {
    if (j < nch) {
      int p = j * 64 + lane;
      bool valid = p < sx;
      CC l = valid ? cc[base + p] : CC(0);
      CC prev = shfl_up_any(l, 1);
      if (lane == 0) prev = tail;
      bool start = valid && (p == 0 || prev != l);
      unsigned long long S = __ballot(start);
      unsigned long long below = S & lanes_upto(lane);
      cst[j] = below ? j * 64 + 63 - __clzll((long long)below) : carry;
      if (S) carry = j * 64 + 63 - __clzll((long long)S);
      lab[j] = l;
      tail = CC(__shfl((unsigned long long)l, 63, 64));
    }
  }
  int carry_d = sx - 1;
  CC head = CC(0);
#pragma unroll
  for (int jj = MAXCH - 1; jj >= 0; --jj) {
    if (jj < nch) {
      int p = jj * 64 + lane;
      bool valid = p < sx;
      CC l = lab[jj];
      CC next = CC(__shfl_down((unsigned long long)l, 1, 64));
      if (lane == 63) next = head;
      bool end = valid && (p == sx - 1 || next != l);
      unsigned long long E = __ballot(end);
      unsigned long long above = lane == 0 ? E : (E & ~((1ULL << lane) - 1ULL));
      int dd = above ? jj * 64 + __ffsll((long long)above) - 1 : carry_d;
      if (E) carry_d = jj * 64 + __ffsll((long long)E) - 1;
      head = CC(__shfl((unsigned long long)l, 0, 64));
      if (valid && l != CC(0)) {
        int c = cst[jj];
        float best = kInf;
        if (c > 0 || bb) { float t = acc[p - c + 1]; best = t * t; }
        if (dd < sx - 1 || bb) { float t = acc[dd + 1 - p]; float v = t * t; if (v < best) best = v; }
        D[base + p] = best;
      }
    }
  }
}

// Serial x pass for rows longer than the wave path handles (one thread per row).
template <class CC>
__global__ void __launch_bounds__(256) edt_x_serial(const CC *cc, int sx, int rows, const float *acc, int bb, float *D) {
  int row = blockIdx.x * 256 + threadIdx.x;
  if (row >= rows) return;
  long long base = (long long)row * sx;
  int i = 0;
  while (i < sx) {
    CC l = cc[base + i];
    int c = i, d = i;
    while (d + 1 < sx && cc[base + d + 1] == l) d++;
    if (l != CC(0))
      for (int p = c; p <= d; ++p) {
        float best = kInf;
        if (c > 0 || bb) { float t = acc[p - c + 1]; best = t * t; }
        if (d < sx - 1 || bb) { float t = acc[d + 1 - p]; float v = t * t; if (v < best) best = v; }
        D[base + p] = best;
      }
    i = d + 1;
  }
}

// Lower envelopes along y (axis 1) or z (axis 2) for lines too long for LDS, run-parallel. A run is a maximal stretch of one
// nonzero id along a line; runs are independent (the walls at their ends stand for the
// neighbouring id or the border), so each run gets its own thread and no wave waits on another
// line's runs.
//   edt_runs:   one thread per line: lists the line's runs (count-only when runs == nullptr) and
//               writes the background zeros of the last pass;
//   edt_run_fh: one thread per run: the envelope of the run's parabolas (heights from the previous
//               pass) with float64 intersections, then the run's values.
// The envelope stack keeps its first kRunStack entries in LDS; deeper stacks spill to a per-run
// global column. The intersection of entries j-1 and j is recomputed from them when needed -- the
// same expression on the same operands as when entry j was placed, so the same bits.
constexpr int kRunStack = 24, kRunBlock = 256, kLineChunk = 8;

struct LineGeom {
  long long base, stride;
  int n;
};
__device__ __forceinline__ LineGeom line_geom(Dims dm, int axis, int t) {
  LineGeom g;
  if (axis == 1) {
    const int x = t % dm.sx, z = t / dm.sx;
    g.base = x + (long long)dm.sx * dm.sy * z;
    g.n = dm.sy;
    g.stride = dm.sx;
  } else {
    g.base = t;
    g.n = dm.sz;
    g.stride = (long long)dm.sx * dm.sy;
  }
  return g;
}

// Run record: x = line, y = first position, z = last position | left wall << 29 | right wall << 30,
// w = first entry of the run's spill column. The count pass stores each line's number of runs and
// of spill entries; the list pass writes the line's runs from the scanned offsets (no shared
// counters).
template <class CC>
__global__ void __launch_bounds__(256) edt_runs(const CC *cc, Dims dm, int axis, int bb, int nlines, int finish, float *D,
                                                int *line_runs, long long *line_spill, const int *run_at,
                                                const long long *spill_at, int4 *runs) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= nlines) return;
  const LineGeom g = line_geom(dm, axis, t);
  const bool list = runs != nullptr;
  int nr = 0;
  long long ns = 0, at = list ? spill_at[t] : 0;
  const int first = list ? run_at[t] : 0;
  auto emit = [&](int c, int d, bool right) {
    const int spill = max(0, d - c + 3 - kRunStack);
    if (list) runs[first + nr] = make_int4(t, c, d | ((c > 0 || bb) ? 1 << 29 : 0) | (right ? 1 << 30 : 0), int(at + ns));
    ++nr;
    ns += spill;
  };
  CC cur = CC(0);
  int c = 0;
  for (int y0 = 0; y0 < g.n; y0 += kLineChunk) {
    CC lab[kLineChunk];
#pragma unroll
    for (int j = 0; j < kLineChunk; ++j) lab[j] = y0 + j < g.n ? cc[g.base + (y0 + j) * g.stride] : CC(0);
    const int m = min(kLineChunk, g.n - y0);
    for (int j = 0; j < m; ++j) {
      const int y = y0 + j;
      const CC l = lab[j];
      if (l != cur) {
        if (cur != CC(0)) emit(c, y - 1, true);
        c = y;
        cur = l;
      }
      if (l == CC(0) && finish && list) D[g.base + y * g.stride] = 0.0f;
    }
  }
  if (cur != CC(0)) emit(c, g.n - 1, bb != 0);
  if (!list) {
    line_runs[t] = nr;
    line_spill[t] = ns;
  }
}

template <class CC>
__global__ void __launch_bounds__(kRunBlock) edt_run_fh(const CC *cc, Dims dm, int axis, float w, int nruns,
                                                        const int4 *runs, int *spill_v, float *spill_h, float *D,
                                                        int finish, unsigned *label_max) {
  __shared__ int sV[kRunStack * kRunBlock];
  __shared__ float sH[kRunStack * kRunBlock];
  const int tid = threadIdx.x;
  const int i = blockIdx.x * kRunBlock + tid;
  if (i >= nruns) return;
  const int4 r = runs[i];
  const LineGeom g = line_geom(dm, axis, r.x);
  const int c = r.y, d = r.z & ((1 << 29) - 1);
  const bool left = (r.z >> 29) & 1, right = (r.z >> 30) & 1;
  int *sv = spill_v + r.w;
  float *sh = spill_h + r.w;
  const double w2 = (double)(w * w);
  auto getV = [&](int k) -> int { return k < kRunStack ? sV[k * kRunBlock + tid] : sv[k - kRunStack]; };
  auto getH = [&](int k) -> float { return k < kRunStack ? sH[k * kRunBlock + tid] : sh[k - kRunStack]; };
  auto set = [&](int k, int v, float h) {
    if (k < kRunStack) { sV[k * kRunBlock + tid] = v; sH[k * kRunBlock + tid] = h; }
    else { sv[k - kRunStack] = v; sh[k - kRunStack] = h; }
  };
  // intersection of entries j-1 and j (j >= 1), as computed when entry j was placed
  auto inter = [&](int j) -> double {
    double v1 = (double)getV(j - 1), h1 = (double)getH(j - 1), v2 = (double)getV(j), h2 = (double)getH(j);
    return ((h2 + w2 * v2 * v2) - (h1 + w2 * v1 * v1)) / (2.0 * w2 * (v2 - v1));
  };
  int k = -1;
  auto place = [&](int pp, double ph) {
    bool placed = false;
    while (k >= 0 && !placed) {
      double vk = (double)getV(k), hk = (double)getH(k);
      double s = ((ph + w2 * (double)pp * (double)pp) - (hk + w2 * vk * vk)) / (2.0 * w2 * ((double)pp - vk));
      double zk = k == 0 ? -1e300 : inter(k);
      if (s <= zk) {
        k--;
      } else {
        k++;
        set(k, pp, (float)ph);
        placed = true;
      }
    }
    if (!placed) { k = 0; set(0, pp, (float)ph); }
  };
  if (left) { k = 0; set(0, c - 1, 0.0f); }
  for (int q0 = c; q0 <= d; q0 += kLineChunk) {  // heights of the previous pass, a chunk in flight
    float hv[kLineChunk];
#pragma unroll
    for (int j = 0; j < kLineChunk; ++j) hv[j] = q0 + j <= d ? D[g.base + (q0 + j) * g.stride] : kInf;
    const int m = min(kLineChunk, d - q0 + 1);
    for (int j = 0; j < m; ++j)
      if (hv[j] < kInf) place(q0 + j, (double)hv[j]);
  }
  if (right) place(d + 1, 0.0);
  float run_max = 0.0f;
  if (k < 0) {
    for (int q = c; q <= d; ++q) D[g.base + q * g.stride] = kInf;
    run_max = kInf;
  } else {
    int kk = 0;
    double znext = k >= 1 ? inter(1) : 0.0;
    int vkk = getV(0);
    float hkk = getH(0);
    for (int q = c; q <= d; ++q) {
      while (kk < k && znext < (double)q) {
        kk++;
        vkk = getV(kk);
        hkk = getH(kk);
        if (kk < k) znext = inter(kk + 1);
      }
      double dq = (double)q - (double)vkk;
      float v = (float)(w2 * dq * dq + (double)hkk);
      if (finish) { v = sqrtf(v); run_max = fmaxf(run_max, v); }
      D[g.base + q * g.stride] = v;
    }
  }
  if (finish && label_max && run_max < kInf) {
    unsigned bits = __float_as_uint(run_max);
    unsigned *slot = label_max + (unsigned long long)cc[g.base + c * g.stride];
    if (ld_u(slot) < bits) atomicMax(slot, bits);
  }
}

// Lower envelopes along y (axis 1) or z (axis 2) in LDS: a block takes XT neighbouring lines whole,
// its lane l = thread % XT their l-th, and finds for every voxel the nearest vertex of its run (the
// position whose height plus squared distance is least, the walls at the run's ends being vertices of
// height 0) by halving: nearest vertices move monotonically along a run, so a row's vertex lies between
// those of the rows around it. Rows at multiples of 16 search outward until the distance alone is too far;
// rows halfway between known ones search between the two vertices, at steps 8 and 4; the
// four rows from each of those then share one pass over the candidates up to the next: some ten
// candidates per voxel whatever the distances are.
// The envelope of the long-line path gives the same values: w2 has a float's 24 bits and a distance
// at most 13, so w2 * dq * dq is exact in float64 (and the fused sums below round once, as its
// separate ones do), the least of the sums is the envelope's value, and candidates that tie give the
// same bits.
// LDS per line and position: 4 bytes of height, a start and a foreground bit, and a 16-bit vertex for
// every fourth row. Four blocks to a compute unit (kLineLds and the registers allow that), so that
// some load while others search. Every voxel is read once and written once, rows of XT at a time; a
// thread per run instead (runs in line order, each lane at its own row, an intersection's division or
// two per step) took 2 x (1.08 + 0.20) ms for 450 x 387 x 256 16-bit cells; y 0.44 and z 0.27 now, bound by
// instructions (some 300 per row of a wave, half of them in float64). A solid 512^3 volume with a black
// border: 26.8 -> 5.1 ms. Searching outward from every 64th row and halving from 32 is 4 % slower on cells.
constexpr int kLineThreads = 256, kSeed = 16;
constexpr size_t kLineLds = 40 << 10, kLineLdsMost = 156 << 10;
constexpr int kWall = 1 << 15;

constexpr size_t line_bytes(int xt, long long n) {
  return size_t(xt) * (size_t(n + 4) * 4 + size_t((n >> 5) + 2) * 8 + size_t((n >> 2) + 2) * 2);
}

// The smaller of two numbers (fmin would first canonicalise what the loop carries).
__device__ __forceinline__ double least(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// A block's lines: heights, start and foreground bits, vertices; l is the lane's line of the XT.
// A vertex is its position + 1, from 0 for the wall before row 0 to n + 1 for the one after the last;
// a vertex code has kWall too for a wall.
template <int XT> struct Line {
  float *h;  // by vertex, and one more that a loop may load ahead
  unsigned *start, *fg, *finite;  // finite: whether any height of the line is
  uint16_t *near;
  int l, n;
  double w2, per_w2;  // the squared step and its inverse
  bool bb;

  __device__ __forceinline__ unsigned start_word(int k) const { return start[k * XT + l]; }
  __device__ __forceinline__ bool foreground(int q) const { return fg[(q >> 5) * XT + l] >> (q & 31) & 1; }

  // The starts at q, q-1, ... (bit 63 first, 32 valid bits) and at q+1, q+2, ... (bit 0 first, 32).
  __device__ __forceinline__ unsigned long long starts_down(int q) const {
    const int k = q >> 5;
    const unsigned long long v = (unsigned long long)start_word(k) << 32 | (k ? start_word(k - 1) : 0u);
    return v << (31 - (q & 31));
  }
  __device__ __forceinline__ unsigned long long starts_up(int q) const {
    const int k = q >> 5;
    const unsigned long long v = (unsigned long long)start_word(k + 1) << 32 | start_word(k);
    return v >> (q & 31) >> 1;
  }
  // The codes of the first and last vertex of run [c, d]: its walls, or its ends where the volume's
  // border is none.
  __device__ __forceinline__ int first_code(int c) const { return c > 0 || bb ? c | kWall : c + 1; }
  __device__ __forceinline__ int last_code(int d) const { return d + 1 < n || bb ? (d + 2) | kWall : d + 1; }

  // The vertices between two codes of a run, in either order.
  struct Range {
    int lo, hi, first, last;  // vertices; the first and last that are no walls
  };
  __device__ __forceinline__ Range range(int a, int b) const {
    const int x = min(a & (kWall - 1), b & (kWall - 1)), y = max(a & (kWall - 1), b & (kWall - 1));
    const bool wx = (x == (a & (kWall - 1)) ? a : b) & kWall, wy = (y == (b & (kWall - 1)) ? b : a) & kWall;
    return Range{x, y, x + int(wx), y - int(wy)};
  }
  __device__ __forceinline__ float stored(int v) const { return h[v * XT + l]; }
  // Vertex v's height from what is stored at its place.
  __device__ __forceinline__ static double height(float value, int v, const Range &r) {
    return double(v < r.first || v > r.last ? 0.0f : value);
  }
  __device__ __forceinline__ double cost(int q, int code) const {
    const int v = code & (kWall - 1);
    const double dq = double(q + 1 - v);
    return __builtin_fma(w2 * dq, dq, code & kWall ? 0.0 : double(h[v * XT + l]));
  }

  // The code of row q's best vertex between codes a and b.
  __device__ __forceinline__ int between(int q, int a, int b) const {
    const Range r = range(a, b);
    double dq = double(q + 1 - r.lo);
    double best = __builtin_fma(w2 * dq, dq, height(stored(r.lo), r.lo, r));
    int vertex = r.lo, v = r.lo + 1, hi = r.hi;
    if (hi - v > 6) {  // none beyond the distance that alone costs as much (in rows: a float of any step's size)
      const int reach = int(fminf(__builtin_amdgcn_sqrtf(float(best * per_w2)) * 1.0001f + 2.0f, float(n)));
      hi = min(hi, q + 1 + reach);
      v = max(v, q + 1 - reach);
      dq = double(q + 2 - v);
    }
    float value = stored(min(v, hi));
    for (; v <= hi; ++v) {
      const float next = stored(v + 1);
      dq -= 1.0;
      const double c = __builtin_fma(w2 * dq, dq, height(value, v, r));
      if (c < best) {
        best = c;
        vertex = v;
      }
      value = next;
    }
    return vertex < r.first || vertex > r.last ? vertex | kWall : vertex;
  }

  // The code of row q's best vertex in run [c, d], outward until the distance alone costs more.
  __device__ __forceinline__ int outward(int q, int c, int d) const {
    const Range r = range(first_code(c), last_code(d));
    int vertex = q + 1;
    double best = double(h[vertex * XT + l]), dr = 1.0;
    const int left = vertex - r.lo, right = r.hi - vertex, most = max(left, right);
    float below = stored(max(q, 0)), above = stored(min(q + 2, n + 1));
    for (int i = 1; i <= most; ++i, dr += 1.0) {
      const double t = w2 * dr * dr;
      if (t >= best) break;
      const int x = q + 1 - i, y = q + 1 + i;
      const float next_below = stored(max(x - 1, 0)), next_above = stored(min(y + 1, n + 1));
      const double cx = t + height(below, x, r), cy = t + height(above, y, r);
      if (i <= left && cx < best) {
        best = cx;
        vertex = x;
      }
      if (i <= right && cy < best) {
        best = cy;
        vertex = y;
      }
      below = next_below;
      above = next_above;
    }
    return vertex < r.first || vertex > r.last ? vertex | kWall : vertex;
  }
};

template <class CC, int XT>
__global__ void __launch_bounds__(kLineThreads, 4) edt_lines(const CC *cc, Dims dm, int axis, float w, int bb, int nlines, int tiles,
                                                             int finish, float *D, unsigned *label_max) {
  extern __shared__ float edt_lds[];
  constexpr int kRows = kLineThreads / XT;  // rows, words or groups of rows that the block takes at a time
  // neighbouring tiles to one XCD: they share the cache lines at their edges
  const int per = (tiles + 7) >> 3, tile = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
  if (tile >= tiles) return;  // whole block
  const int l = threadIdx.x % XT, row = threadIdx.x / XT, t = tile * XT + l;
  const LineGeom g = line_geom(dm, axis, t < nlines ? t : 0);
  const int n = g.n, words = (n >> 5) + 2;
  Line<XT> a;
  a.h = edt_lds;
  a.start = reinterpret_cast<unsigned *>(edt_lds + XT * (n + 3));
  a.fg = a.start + XT * words;
  a.finite = a.fg + XT * words;
  a.near = reinterpret_cast<uint16_t *>(a.finite + XT);
  a.l = l;
  a.n = n;
  a.w2 = double(w * w);
  a.per_w2 = 1.0 / a.w2;
  a.bb = bb != 0;

  if (row == 0) a.finite[l] = 0;
  unsigned any = 0, inner = 0;  // foreground; starts within the line
  for (int k = row; k < words; k += kRows) {
    unsigned start = 0, fg = 0;
    if (t < nlines && k * 32 < n) {
      const CC *at = cc + g.base + (long long)(k * 32) * g.stride;
      CC prev = k ? at[-g.stride] : CC(0);
#pragma unroll 1
      for (int j0 = 0; j0 < 32; j0 += 16) {
        CC lab[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) lab[j] = k * 32 + j0 + j < n ? at[(j0 + j) * g.stride] : CC(0);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          start |= unsigned(lab[j] != prev) << (j0 + j);
          fg |= unsigned(lab[j] != CC(0)) << (j0 + j);
          prev = lab[j];
        }
      }
    }
    const int left = n - k * 32;
    inner |= start & (left >= 32 ? ~0u : left > 0 ? (1u << left) - 1u : 0u) & (k == 0 ? ~1u : ~0u);
    if (k == 0) start |= 1u;                   // row 0
    if (k == n >> 5) start |= 1u << (n & 31);  // the end of the last run
    a.start[k * XT + l] = start;
    a.fg[k * XT + l] = fg;
    any |= fg;
  }
  const bool some = __syncthreads_or(int(any != 0));
  if (!some) {
    if (finish && t < nlines)
      for (int q = row; q < n; q += kRows) D[g.base + q * g.stride] = 0.0f;
    return;
  }
  constexpr int kLoads = 8;
  bool finite = false;
  for (int q0 = row; q0 < n; q0 += kLoads * kRows) {
    float value[kLoads];
    unsigned fg = 0;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int q = q0 + j * kRows;
      const bool f = q < n && a.foreground(q);
      fg |= unsigned(f) << j;
      value[j] = D[g.base + (f ? q : 0) * g.stride];  // the line's first row stands in for one not needed
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int q = q0 + j * kRows;
      if (fg >> j & 1) {
        a.h[(q + 1) * XT + l] = value[j];
        finite |= value[j] < kInf;
      }
      if (finish && !(fg >> j & 1) && q < n && t < nlines) D[g.base + q * g.stride] = 0.0f;
    }
  }
  if (finite) a.finite[l] = 1;
  if (!__syncthreads_or(int(finite || inner || bb))) {  // no wall and no height in the block's lines
    for (int q = row; q < n; q += kRows)
      if (a.foreground(q)) D[g.base + q * g.stride] = kInf;
    return;
  }
  for (int q = row * kSeed; q < n; q += kRows * kSeed) {
    if (!a.foreground(q)) continue;
    int k = q >> 5;
    unsigned v = a.start_word(k) & ((2u << (q & 31)) - 1u);
    while (!v) v = a.start_word(--k);  // row 0 has one
    const int c = k * 32 + 31 - __clz(int(v));
    k = q >> 5;
    v = a.start_word(k) & ~((2u << (q & 31)) - 1u);
    while (!v) v = a.start_word(++k);  // n has one
    const int d = k * 32 + __ffs(int(v)) - 2;
    // a whole line without walls and heights has nothing to search for
    const bool none = c == 0 && d == n - 1 && !bb && !a.finite[l];
    a.near[(q >> 2) * XT + l] = uint16_t(none ? q + 1 : a.outward(q, c, d));
  }
  for (int s = kSeed / 2; s >= 4; s >>= 1) {
    __syncthreads();
    for (int q = s + row * 2 * s; q < n; q += kRows * 2 * s) {
      if (!a.foreground(q)) continue;
      // the vertices of rows q - s and q + s where the run has those, else its first and last
      const unsigned long long down = a.starts_down(q) >> (64 - s) << (64 - s), up = a.starts_up(q) & ((1ULL << s) - 1ULL);
      const int before = down ? a.first_code(q - __clzll((long long)down)) : int(a.near[((q - s) >> 2) * XT + l]);
      const int after = up ? a.last_code(q + __ffsll((long long)up) - 1) : int(a.near[((q + s) >> 2) * XT + l]);
      a.near[(q >> 2) * XT + l] = uint16_t(a.between(q, before, after));
    }
  }
  __syncthreads();
  for (int q0 = 4 * row; q0 < n; q0 += 4 * kRows) {
    const unsigned fg = a.fg[(q0 >> 5) * XT + l] >> (q0 & 31) & 15u;
    if (!fg) continue;
    const unsigned starts = unsigned(a.starts_up(q0)) & 15u;  // at q0 + 1 .. q0 + 4
    const int v0 = a.near[(q0 >> 2) * XT + l], v4 = a.near[((q0 + 4) >> 2) * XT + l];
    double best[4] = {0.0, 0.0, 0.0, 0.0};
    for (int j0 = 0; j0 < 4;) {  // the runs among the four rows, rows j0 to j1 of each
      const unsigned ends = starts >> j0;
      const int j1 = ends ? j0 + __ffs(int(ends)) - 1 : 3;
      if (fg >> j0 & 1) {
        const auto r = a.range(j0 ? a.first_code(q0 + j0) : v0, ends ? a.last_code(q0 + j1) : v4);
        double m[4] = {HUGE_VAL, HUGE_VAL, HUGE_VAL, HUGE_VAL}, dq = double(q0 + 1 - r.lo);
        float stored = a.stored(r.lo);
        for (int v = r.lo; v <= r.hi; ++v) {
          const float next = a.stored(v + 1);
          const double h = a.height(stored, v, r);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const double x = dq + double(j);
            m[j] = least(m[j], __builtin_fma(a.w2 * x, x, h));
          }
          dq -= 1.0;
          stored = next;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j >= j0 && j <= j1) best[j] = m[j];
      }
      j0 = j1 + 1;
    }
    float *out = D + g.base + q0 * g.stride;
    float value[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      value[j] = float(best[j]);
      if (finish) value[j] = sqrtf(value[j]);
      if (fg >> j & 1) out[j * g.stride] = value[j];
    }
    if (!finish || !label_max) continue;
    // Each run's largest value among these rows goes to its label's maximum, unless the run goes on to
    // a row q0 + 4 as large or came from a larger row q0 - 4: the groups that hold a run's maximum
    // include a last one, which neither rule leaves out.
    float top = 0.0f;
    bool open = q0 && !(a.starts_down(q0) >> 60);  // the first run is that of q0 - 4
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      top = fmaxf(top, value[j]);
      const bool ends = starts >> j & 1;
      if ((ends || j == 3) && (fg >> j & 1) && top < kInf) {
        bool tell = true;
        if (!ends) tell = sqrtf(float(a.cost(q0 + 4, v4))) < top;
        if (open && tell) tell = sqrtf(float(a.cost(q0 - 4, a.near[((q0 - 4) >> 2) * XT + l]))) <= top;
        if (tell) {
          unsigned *slot = label_max + (unsigned long long)cc[g.base + (q0 + j) * g.stride];
          const unsigned bits = __float_as_uint(top);
          if (ld_u(slot) < bits) atomicMax(slot, bits);
        }
      }
      if (ends) {
        top = 0.0f;
        open = false;
      }
    }
  }
}

template <class CC, int XT>
void run_lines(Context &ctx, const CC *cc, Dims dm, int axis, float w, bool bb, int nlines, int n, bool finish, float *out,
               unsigned *label_max) {
  const size_t lds = line_bytes(XT, n);
  if (lds > (64 << 10))
    BROOK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(edt_lines<CC, XT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(kLineLdsMost)));
  const int tiles = (nlines + XT - 1) / XT;
  edt_lines<CC, XT><<<unsigned((tiles + 7) / 8 * 8), kLineThreads, lds, ctx.stream()>>>(cc, dm, axis, w, bb, nlines, tiles, finish,
                                                                                       out, label_max);
  BROOK_LAUNCHED();
}

// finish for a single pass (x only): background 0, else sqrt.
template <class CC>
__global__ void __launch_bounds__(256) edt_finish(const CC *cc, long long n, float *D, unsigned *label_max) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  CC l = cc[i];
  if (l == CC(0)) { D[i] = 0.0f; return; }
  float v = sqrtf(D[i]);
  D[i] = v;
  if (label_max && v < kInf) atomicMax(label_max + (unsigned long long)l, __float_as_uint(v));
}

template <class CC>
void run_edt(Context &ctx, const CC *cc, Dims dm, const float aniso[3], bool bb, int dims_used, float *out,
             unsigned *label_max) {
  auto s = ctx.stream();
  const int rows = dm.sy * dm.sz;
  std::vector<float> table(dm.sx + 2, 0.0f);
  for (size_t k = 1; k < table.size(); ++k) table[k] = table[k - 1] + aniso[0];
  Buffer<float> acc(ctx, table.size());
  acc.upload(ctx, table.data(), table.size());
  {
    KernelTimer x_timer(ctx, "edt_x");
    if (dm.sx <= 128)
      edt_x<CC, 2><<<(rows + 3) / 4, 256, 0, s>>>(cc, dm.sx, rows, acc.data(), bb, out);
    else if (dm.sx <= 512)
      edt_x<CC, 8><<<(rows + 3) / 4, 256, 0, s>>>(cc, dm.sx, rows, acc.data(), bb, out);
    else if (dm.sx <= 2048)
      edt_x<CC, 32><<<(rows + 3) / 4, 256, 0, s>>>(cc, dm.sx, rows, acc.data(), bb, out);
    else
      edt_x_serial<CC><<<(rows + 255) / 256, 256, 0, s>>>(cc, dm.sx, rows, acc.data(), bb, out);
    BROOK_LAUNCHED();
  }
  const int last = dims_used - 1;
  if (last == 0) {
    long long n = (long long)dm.sx * dm.sy * dm.sz;
    edt_finish<CC><<<unsigned((n + 255) / 256), 256, 0, s>>>(cc, n, out, label_max);
    BROOK_LAUNCHED();
    return;
  }
  for (int axis = 1; axis <= last; ++axis) {
    const int nlines = axis == 1 ? dm.sx * dm.sz : dm.sx * dm.sy;
    const unsigned lgrid = unsigned((nlines + 255) / 256);
    const char *timer = axis == 1 ? "edt_y" : "edt_z";
    const int n = axis == 1 ? dm.sy : dm.sz;
    const float w = aniso[axis];
    // As many lines to a block as leave room for three others on the compute unit (kLineLds), down to the 8
    // whose rows still fill 32-byte sectors: those have up to all of its LDS, and longer lines take the run
    // lists. Lines of up to 27 positions go to a thread each, 256 to a block: with 32 lines most threads had no
    // row (z of 9000 x 9000 x 1 8.67 ms, now 1.80, the run lists 2.93; of 4000 x 4000 x 4 1.96, 0.41, 1.02;
    // of 2000 x 2000 x 27 1.01, 0.53, 1.14). 64 or 128 lines were slower up to 27 (4.34, 2.67 ms; 0.62, 0.53).
    if (line_bytes(8, n) <= kLineLdsMost) {
      KernelTimer line_timer(ctx, timer);
      if (line_bytes(kLineThreads, n) <= kLineLds) run_lines<CC, kLineThreads>(ctx, cc, dm, axis, w, bb, nlines, n, axis == last, out, label_max);
      else if (line_bytes(32, n) <= kLineLds) run_lines<CC, 32>(ctx, cc, dm, axis, w, bb, nlines, n, axis == last, out, label_max);
      else if (line_bytes(16, n) <= kLineLds) run_lines<CC, 16>(ctx, cc, dm, axis, w, bb, nlines, n, axis == last, out, label_max);
      else run_lines<CC, 8>(ctx, cc, dm, axis, w, bb, nlines, n, axis == last, out, label_max);
      continue;
    }
    // (two timer scopes below: the host read between them is not timed)
    Buffer<int> line_runs(ctx, size_t(nlines)), run_at(ctx, size_t(nlines));
    Buffer<long long> line_spill(ctx, size_t(nlines)), spill_at(ctx, size_t(nlines));
    {
      KernelTimer count_timer(ctx, timer);
      edt_runs<CC><<<lgrid, 256, 0, s>>>(cc, dm, axis, bb, nlines, 0, out, line_runs.data(), line_spill.data(), nullptr,
                                         nullptr, nullptr);
      BROOK_LAUNCHED();
      exclusive_sum(ctx, line_runs.data(), run_at.data(), nlines);
      exclusive_sum(ctx, line_spill.data(), spill_at.data(), nlines);
    }
    int last_runs = 0, last_at = 0;
    long long last_spill = 0, last_spill_at = 0;
    BROOK_HIP(hipMemcpyAsync(&last_runs, line_runs.data() + nlines - 1, 4, hipMemcpyDeviceToHost, s));
    BROOK_HIP(hipMemcpyAsync(&last_at, run_at.data() + nlines - 1, 4, hipMemcpyDeviceToHost, s));
    BROOK_HIP(hipMemcpyAsync(&last_spill, line_spill.data() + nlines - 1, 8, hipMemcpyDeviceToHost, s));
    BROOK_HIP(hipMemcpyAsync(&last_spill_at, spill_at.data() + nlines - 1, 8, hipMemcpyDeviceToHost, s));
    ctx.synchronize();
    const long long total_runs = (long long)last_at + last_runs, total_spill = last_spill_at + last_spill;
    if (total_runs > INT32_MAX || total_spill > INT32_MAX)
      throw Unsupported("EDT envelope spill exceeds 2^31 entries (runs too long for this build)");
    const int nruns = int(total_runs);
    Buffer<int4> runs(ctx, size_t(std::max(nruns, 1)));
    Buffer<int> V(ctx, size_t(std::max<long long>(total_spill, 1)));
    Buffer<float> H(ctx, size_t(std::max<long long>(total_spill, 1)));
    KernelTimer fh_timer(ctx, timer);
    edt_runs<CC><<<lgrid, 256, 0, s>>>(cc, dm, axis, bb, nlines, axis == last, out, nullptr, nullptr, run_at.data(),
                                       spill_at.data(), runs.data());
    BROOK_LAUNCHED();
    if (nruns) {
      edt_run_fh<CC><<<unsigned((nruns + kRunBlock - 1) / kRunBlock), kRunBlock, 0, s>>>(
          cc, dm, axis, aniso[axis], nruns, runs.data(), V.data(), H.data(), out, axis == last, label_max);
      BROOK_LAUNCHED();
    }
  }
}

}  // namespace

void edt(Context &ctx, const void *cc, int cc_bytes, Dims dims, const float aniso[3], bool black_border, int dims_used,
         float *out, unsigned *label_max) {
  for (int a = 0; a < 3; ++a)
    if (!(aniso[a] > 0) || !std::isfinite(aniso[a])) throw std::invalid_argument("anisotropy must be finite and positive");
  if (int64_t(dims.sx) * dims.sy * dims.sz == 0) return;
  if (cc_bytes == 1) run_edt<uint8_t>(ctx, static_cast<const uint8_t *>(cc), dims, aniso, black_border, dims_used, out, label_max);
  else if (cc_bytes == 2) run_edt<uint16_t>(ctx, static_cast<const uint16_t *>(cc), dims, aniso, black_border, dims_used, out, label_max);
  else run_edt<uint32_t>(ctx, static_cast<const uint32_t *>(cc), dims, aniso, black_border, dims_used, out, label_max);
}

}  // namespace brook
