// The quotient by the divisor's reciprocal and two correction steps, as the
// affine quantizer and the codec's unit vectors form it, against the division:
// random operands, quotients at and beside ties of whole numbers, and exact
// multiples, with divisors whose mantissa is not all ones.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

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
  std::mt19937_64 rng(1);
  long bad = 0, n = 0;
  for (int i = 0; i < 12000000; i++) {
    const uint64_t r = rng();
    // a divisor in [2^-60, 2^20]
    uint32_t m = static_cast<uint32_t>(r) & 0x7fffffu;
    if (m == 0x7fffffu) continue;
    if ((r >> 60) == 0) m = 0x7ffffeu - static_cast<uint32_t>(r >> 50 & 15);  // nearly all ones
    const float den = bits(static_cast<uint32_t>(127 - 60 + (r >> 23) % 81) << 23 | m);
    float x;
    switch ((r >> 32) & 3) {
      case 0:  // a random mantissa, within 2^+-8 of the divisor
        x = bits(static_cast<uint32_t>(r >> 34) & 0x7fffffu | 0x3f800000u) * den *
            std::ldexp(1.0f, static_cast<int>(r >> 57 & 15) - 8);
        break;
      case 1:  // at a tie of two whole numbers
        x = den * (static_cast<float>(r >> 34 & 255) + 0.5f);
        break;
      case 2:  // one unit beside it
        x = bits(bits(den * (static_cast<float>(r >> 34 & 255) + 0.5f)) + ((r >> 44 & 1) ? 1u : -1u));
        break;
      default: x = den * static_cast<float>(r >> 34 & 255);
    }
    const float inv = 1.0f / den;
    float q = x * inv;
    q = fmaf(fmaf(-q, den, x), inv, q);
    q = fmaf(fmaf(-q, den, x), inv, q);
    n++;
    if (q != x / den && bad++ < 5) std::printf("%a / %a: %a, not %a\n", x, den, q, x / den);
    // round half away of a non-negative quotient below 2^22
    if (static_cast<uint32_t>(q + 0.49999997f) != static_cast<uint32_t>(std::round(x / den)) && bad++ < 5)
      std::printf("code of %a\n", q);
  }
  std::printf("%ld pairs, %ld differ\n", n, bad);
  return bad != 0;
}
