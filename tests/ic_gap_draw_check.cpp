// Host check that ic_gap_draw (double precision with an integer fallback)
// gives ic_gap's value: for q of every threshold class a row can have, at
// uniforms on both sides of gap boundaries (where rounding could decide), at
// the ends of the range and at random.
// Usage: ic_gap_draw_check <seed> <rows>; prints "ok" and exits 0 when all agree.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../ripples_amd/csrc/ic_gap.h"

using namespace rip;

int main(int argc, char **argv) {
  const unsigned seed = argc > 1 ? std::atoi(argv[1]) : 1;
  const int rows = argc > 2 ? std::atoi(argv[2]) : 1000;
  std::mt19937_64 rng(seed);
  IcGapTab tab;
  for (uint32_t i = 0; i < 256; ++i) ic_gap_tab_entry(&tab, i);
  int fails = 0;
  uint64_t checked = 0;
  for (int r = 0; r < rows; ++r) {
    uint32_t T;
    switch (r % 7) {
      case 0: T = 1 + static_cast<uint32_t>(rng() % 64); break;
      case 1: T = (1u << 24) - static_cast<uint32_t>(rng() % 64); break;   // 2^24 among them: q = 0
      case 2: T = (1u << 23) + static_cast<uint32_t>(rng() % 129) - 64; break;
      case 3: T = 1u << (rng() % 24); break;
      case 4: T = (1u << 24) / (1 + static_cast<uint32_t>(rng() % 5000)); break;   // 1 / indegree
      default: T = 1 + static_cast<uint32_t>(rng() % ((1u << 24) - 1)); break;
    }
    const uint64_t q = ic_gap_q(T);
    const double inv = ic_gap_inv(q);
    auto check = [&](uint64_t U) {
      if (U < 1 || U > (1ull << 32)) return;
      const uint64_t x = ((U - 1) << 32) | (rng() & 0xFFFFFFFFull);
      const uint64_t a = ic_gap(x, q), b = ic_gap_draw(x, q, inv, &tab);
      ++checked;
      if (a != b && fails++ < 10)
        std::printf("FAIL T=%u U=%llu %llu %llu\n", T, (unsigned long long)U,
                    (unsigned long long)a, (unsigned long long)b);
    };
    for (uint64_t d = 0; d < 4; ++d) {
      check(1 + d);
      check((1ull << 32) - d);
      check((1ull << (rng() % 33)) + d - 1);   // where the exponent steps
    }
    for (int i = 0; i < 100; ++i) check(1 + rng() % (1ull << 32));
    // gap boundaries: the largest U whose gap reaches len, and its neighbours
    for (int i = 0; i < 12; ++i) {
      const uint64_t u = ic_skip_len(q, 1 + static_cast<uint32_t>(rng() % (1u << (1 + i))));
      for (int d = -1; d <= 2; ++d) check(u + d);
    }
  }
  if (fails || !checked) {
    std::printf("%d failures\n", fails);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
