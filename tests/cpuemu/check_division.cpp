// Every float significand: the refined reciprocal from every seed within one ulp
// of 1 / b (the all-ones significand: from the right one), and quotients of
// pseudo-random numerators, against the IEEE division.
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "division.hpp"

static float bits(uint32_t u) {
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
static uint32_t bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}

int main() {
  long wrong_reciprocals = 0, wrong_quotients = 0;
  uint32_t r = 12345;
  for (uint32_t m = 0; m < 1u << 23; m++) {
    const float b = bits((127u - m % 7) << 23 | m), want = 1.0f / b;
    const bool all_ones = m == (1u << 23) - 1;
    for (int d = all_ones ? 0 : -1; d <= (all_ones ? 0 : 1); d++)
      wrong_reciprocals += sfx::refined_reciprocal(b, bits(bits(want) + d)) != want;
    const float y = sfx::reciprocal(b);
    wrong_reciprocals += y != want;
    for (int n = 0; n < (all_ones ? 100000 : 2); n++) {
      r = r * 1664525u + 1013904223u;
      const float a = bits((r & 0x807fffffu) | (100u + (r >> 8) % 50u) << 23);
      wrong_quotients += sfx::quotient(a, b, y) != a / b;
    }
  }
  std::printf("wrong reciprocals %ld, wrong quotients %ld\n", wrong_reciprocals, wrong_quotients);
  return wrong_reciprocals || wrong_quotients;
}
