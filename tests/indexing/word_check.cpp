// CPU check of the frontier kernels' word and index arithmetic (common.hpp, front.hpp): divisions by
// a high product for divisors and dividends at the edges of their ranges, the lane slots in address
// order, the order of road words of one voxel, the steps and the padding that has to hold them. Prints
// "ok" or the first violation.
#include <cstdio>
#include <initializer_list>

#include "../../brook_amd/csrc/front.hpp"

using namespace brook;

int main() {
  for (unsigned d : {1u, 2u, 3u, 5u, 7u, 48u, 64u, 127u, 128u, 129u, 512u, 641u, 1000u, 4095u, 65535u, 65536u, 65537u, 262144u,
                     1000003u, (1u << 30) - 1u, 1u << 30, (1u << 30) + 1u, (1u << 31) - 1u}) {
    const FastDiv f = fast_div(d);
    auto check = [&](unsigned n) { return fast_quotient(n, f) == n / d; };
    const unsigned top = (1u << 31) - 1u;
    for (unsigned i = 0; i < 3000; ++i)
      for (unsigned n : {i, top - i, unsigned((unsigned long long)i * 715827ull % (1ull << 31))})
        if (!check(n)) { std::printf("%u / %u\n", n, d); return 1; }
    for (unsigned long long q = 1; q * d <= top; q = q * 3 / 2 + 1)  // around multiples of d
      for (int e = -1; e <= 1; ++e)
        if (q * d + e <= top && !check(unsigned(q * d + e))) { std::printf("%llu * %u + %d\n", q, d, e); return 1; }
  }
  const SlotTable t = slot_table();
  bool seen[26] = {};
  for (int s = 0; s < 26; ++s) {
    seen[t.k[s]] = true;
    auto key = [&](int k) { return (kDZ[k] * 1000 + kDY[k]) * 1000 + kDX[k]; };
    if (s && key(t.k[s - 1]) >= key(t.k[s])) { std::printf("slot %d out of order\n", s); return 1; }
  }
  for (bool b : seen)
    if (!b) { std::printf("a neighbour has no slot\n"); return 1; }
  // one voxel's words: by distance, then queued, rail, far-listed; unreached above every finite one
  const unsigned cost = 0x3f800000u, d0 = 0x3f000000u, d1 = d0 + 1u, most = kInfBits - 1u;
  const unsigned long long order[] = {road_word(d0, 0, cost), road_word(d0, kNotQueued, cost),
                                      road_word(d0, kFarListed | kNotQueued, cost), road_word(d1, 0, cost),
                                      road_word(most, kFarListed | kNotQueued, cost), kUnreached | cost};
  for (int i = 1; i < 6; ++i)
    if (order[i - 1] >= order[i]) { std::printf("word %d out of order\n", i); return 1; }
  for (unsigned long long w : order)
    if (road_cost(w) != cost) { std::printf("cost lost\n"); return 1; }
  if (road_dist(kUnreached) != kInfBits || road_dist(order[1]) != d0) { std::printf("distance lost\n"); return 1; }
  // every step of a voxel inside the volume has its flat offset, and every step lies within the padding;
  // a volume of one plane or row is not padded along it
  for (Dims d : {Dims{1, 1, 1}, Dims{7, 1, 1}, Dims{1, 9, 1}, Dims{1, 1, 5}, Dims{6, 5, 1}, Dims{6, 1, 4}, Dims{1, 3, 4}, Dims{5, 4, 3}}) {
    long long longest = 0;
    for (int k = 0; k < 26; ++k) {
      const int off = step_offset(d, kDX[k], kDY[k], kDZ[k]);
      longest = off > longest ? off : longest;
      if (-off > word_pad(d)) { std::printf("step %d beyond the padding\n", k); return 1; }
      const bool stays = (d.sx > 1 || !kDX[k]) && (d.sy > 1 || !kDY[k]) && (d.sz > 1 || !kDZ[k]);  // some voxel has that neighbour
      if (stays && off != kDX[k] + d.sx * (kDY[k] + d.sy * kDZ[k])) { std::printf("step %d of %d %d %d\n", k, d.sx, d.sy, d.sz); return 1; }
    }
    if (longest != word_pad(d)) { std::printf("padding %lld of %d %d %d\n", word_pad(d), d.sx, d.sy, d.sz); return 1; }
  }
  if (word_pad(Dims{4000, 4000, 1}) != 4001) { std::printf("a plane of padding\n"); return 1; }
  std::printf("ok\n");
  return 0;
}
