// The short quotients of the quantiser and of the SiLU epilogue, step by step as the
// kernels write them, against the IEEE quotient.  The hardware's reciprocal is good
// to one unit in the last place: each check runs with the correctly rounded one and
// with its two neighbours.  Prints the number of differences per check.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>

static float f(uint32_t u) { float x; std::memcpy(&x, &u, 4); return x; }
static uint32_t b(float x) { uint32_t u; std::memcpy(&u, &x, 4); return u; }
static float rcp(float d, int off) { return f(b(1.0f / d) + off); }

// 127 / a and a / 127 (linear_small.hip, quantise_row)
static bool quantiser(float a, int off) {
  const float y0 = rcp(a, off), y = std::fmaf(std::fmaf(-a, y0, 1.f), y0, y0);
  float inv = 127.f * y;
  inv = std::fmaf(std::fmaf(-a, inv, 127.f), y, inv);
  const float c = 1.f / 127.f, s0 = a * c, s = std::fmaf(std::fmaf(-127.f, s0, a), c, s0);
  return inv == 127.f / a && s == a / 127.f;
}

// g / d (ovh_common.h, silu_up_lanes)
static bool silu(float g, float d, int off) {
  float y = rcp(d, off);
  y = std::fmaf(std::fmaf(-d, y, 1.f), y, y);
  float q = g * y;
  q = std::fmaf(std::fmaf(-d, q, g), y, q);
  q = std::fmaf(std::fmaf(-d, q, g), y, q);
  return q == g / d;
}

int main() {
  // every significand, at the ends and in the middle of the range of exponents
  const int exps[] = {-100, 0, 119};
  long bad = 0;
  for (uint32_t m = 0; m < 1u << 23; ++m)
    for (int off = -1; off <= 1; ++off) bad += !quantiser(f((127u << 23) | m), off);
  for (int e : exps)
    for (uint32_t m = 0; m < 1u << 23; m += 61)
      for (int off = -1; off <= 1; ++off)
        bad += !quantiser(f(((uint32_t)(127 + e) << 23) | m), off);
  bad += !quantiser(0x1p120f, 0);
  std::printf("quantiser %ld\n", bad);
  // random significands and exponents of g in [2^-100, 2^60] and of d in [1, 2^97)
  // (d beyond 2 only where g is negative, as in 1 + e^-g); then the significands
  // where a quotient's rounding is hardest: d all ones or just above a power of two
  bad = 0;
  uint64_t s = 0x9e3779b97f4a7c15ull;
  auto next = [&] { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; };
  for (long i = 0; i < 20000000; ++i) {
    const uint64_t r = next(), t = next();
    uint32_t mg = r & 0x7fffff, md = (r >> 23) & 0x7fffff;
    if (i % 4 == 1) md = 0x7fffff - (md & 15);
    if (i % 4 == 2) md &= 15;
    if (i % 8 >= 6) mg = (t >> 40) & 1 ? 0x7fffff - (mg & 15) : mg & 15;
    uint32_t ge, de;
    if (t & 1) {  // g < 0: |g| to 66, d to 2^97
      ge = 127 + 6 - (uint32_t)((t >> 8) % 8);
      de = 127 + (uint32_t)((t >> 16) % 97);
    } else {
      ge = 127 - 100 + (uint32_t)((t >> 8) % 161);
      de = 127 + (uint32_t)((t >> 16) % 2);
    }
    const float g = f((ge << 23) | mg | ((uint32_t)(t & 1) << 31)), d = f((de << 23) | md);
    for (int off = -1; off <= 1; ++off) bad += !silu(g, d, off);
  }
  std::printf("silu %ld\n", bad);
  return 0;
}
