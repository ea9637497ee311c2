// The frontier kernels' lane and index arithmetic (front.hpp) on the CPU, run by emulated workgroups:
// a front of any length, with any number of pairs in flight, has each entry served once by each of its 26
// neighbours' lanes and by no other, no wave stages more candidates than its stage holds, and no value
// comes from a lane beyond the wave (the emulation reports that); a lane's byte offset of a word in 32 bits is
// the one in 64 bits and lies in the padded array. Prints "ok" or the first violation.
#include <hip/hip_runtime.h>

#include "common.hpp"
#define wave_slot(counter) emu::slot(counter)
#include "front.hpp"

using namespace brook;

namespace {

int bad = 0;

// Every front length up to `longest` in a workgroup of `block` threads.
template <int Max> void fronts(int block, int longest) {
  const int waves = block / 64;
  const Dims d{1000, 1000, 1000};
  std::vector<int> list(size_t(longest), 0);
  for (int e = 0; e < longest; ++e) list[size_t(e)] = 500000000 + 3 * e;
  std::vector<int> served(size_t(longest) * 32);
  std::vector<Stage> stages(size_t(waves) + 1);
  emu::run(block, emu::Schedule{{}, 3}, [&] {
    const Lane<true> ln = lane_of<true>(d);
    Stage &st = stages[size_t(ln.wave)];
    const SplitList<1 << 30> front{nullptr, list.data()};
    for (int n = 1; n <= longest; ++n) {
      if (threadIdx.x == 0) std::fill(served.begin(), served.end(), 0);
      __syncthreads();
      int staged = 0;
      auto flush = [&](bool all) {
        if (staged > kStage) bad = 1;
        stage_take(st, staged, all, [&](bool on, int, unsigned long long word) {
          if (on) ++served[size_t(word)];
        });
      };
      with_pairs<Max>(n, waves, [&](auto Pairs) {
        constexpr int P = decltype(Pairs)::value;
        for (int b = ln.wave * 2 * P; b < n; b += waves * 2 * P) {
          int u[P];
          const int ue = batch_entries<P>(ln, front, b, n, u);
          const unsigned mine = ln.lane < min(2 * P, n - b) ? (1u << 26) - 1u : 0u;
          staged_pairs<P>([&](int p) {
            const unsigned m = of_entry(ln, mine, 2 * p), entry = of_entry(ln, unsigned(ue), 2 * p);
            if (m && int(entry) != u[p]) bad = 2;
            const int e = (u[p] - 500000000) / 3;
            stage_put(st, staged, (m & ln.bit) != 0u, u[p] + ln.off, (unsigned long long)e * 32 + (unsigned long long)ln.k);
          }, [&] { flush(false); });
        }
      });
      flush(true);
      __syncthreads();
      if (threadIdx.x == 0)
        for (int e = 0; e < longest; ++e)
          for (int k = 0; k < 32; ++k)
            if (served[size_t(e) * 32 + size_t(k)] != int(e < n && k < 26)) {
              std::printf("%d threads, %d pairs, front of %d: entry %d, neighbour %d served %d times\n", block, Max, n, e, k,
                          served[size_t(e) * 32 + size_t(k)]);
              std::fflush(stdout);
              std::_Exit(1);
            }
      __syncthreads();
    }
  });
}

void offsets(Dims d) {
  const long long words = (long long)d.sx * d.sy * d.sz + 2 * word_pad(d), last = (long long)d.sx * d.sy * d.sz - 1;
  emu::run(64, emu::Schedule{{0}, 0}, [&] {
    const Lane<false> narrow = lane_of<false>(d);
    const Lane<true> wide = lane_of<true>(d);
    for (long long u : {0LL, last / 2, last}) {
      const unsigned long long at = wide.at(int(u));
      const int k = narrow.k;
      const long long off = narrow.bit ? step_offset(d, kDX[k], kDY[k], kDZ[k]) : 0;
      if (at != (unsigned long long)(u + off + word_pad(d)) * 8 || at >= (unsigned long long)words * 8) bad = 3;
      if (narrow_words(d) && narrow.at(int(u)) != at) bad = 4;
    }
  });
}

}  // namespace

int main() {
  fronts<9>(64, 70);
  fronts<9>(256, 160);
  fronts<13>(128, 120);
  fronts<26>(128, 240);
  fronts<9>(1024, 300);
  int narrow = 0, wide = 0;
  for (Dims d : {Dims{1, 1, 1}, Dims{5, 1, 1}, Dims{7, 6, 1}, Dims{1, 3, 9}, Dims{512, 512, 512}, Dims{1024, 1024, 509},
                 Dims{1024, 1024, 510}, Dims{1024, 1024, 511}, Dims{9000, 9000, 5}, Dims{23170, 23170, 1}, Dims{1290, 1290, 1290}}) {
    offsets(d);
    (narrow_words(d) ? narrow : wide) += 1;
  }
  if (narrow < 5 || wide < 3) bad = 5;
  if (bad) std::printf("violation %d\n", bad);
  else std::printf("ok\n");
  return bad;
}
