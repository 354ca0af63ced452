// The roundings that the quantizers inside the decode GEMMs take for granted, each over every input it can meet.  Prints the
// mismatches of: the quotient (2^33 pairs), its special case 448, the rounding to whole numbers.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float bits(uint32_t b) {
  float f;
  memcpy(&f, &b, 4);
  return f;
}

int main(void) {
  long quotient = 0, by_448 = 0, whole = 0;
  // one Markstein step on RN(x * RN(1 / s)) against x / s: the 2^10 significands of a 16-bit x (bfloat16 has fewer), the 2^23 of s
#pragma omp parallel for reduction(+ : quotient) schedule(dynamic, 4096)
  for (uint32_t m = 0; m < (1u << 23); m++) {
    const float s = bits(0x3f800000u | m), r = 1.0f / s;
    int bad = 0;
    for (int i = 0; i < 1024; i++) {
      const float x = 1.0f + (float)i / 1024.0f, q = x * r;
      bad += fmaf(fmaf(-q, s, x), r, q) != x / s;
    }
    quotient += bad;
  }
  // the same with s = 448, whose reciprocal is a constant, for every significand of x
#pragma omp parallel for reduction(+ : by_448)
  for (uint32_t m = 0; m < (1u << 23); m++) {
    const float x = bits(0x3f800000u | m), r = 1.0f / 448.0f, q = x * r;
    by_448 += fmaf(fmaf(-q, 448.0f, x), r, q) != x / 448.0f;
  }
  // adding 0.5 less one unit and truncating against roundf: every float of magnitude up to 128
#pragma omp parallel for reduction(+ : whole)
  for (uint32_t b = 0; b <= 0x43000000u; b++) {
    const float q = bits(b);
    whole += (int)(q + 0.49999997f) != (int)roundf(q);
    whole += (int)(-q - 0.49999997f) != (int)roundf(-q);
  }
  printf("%ld %ld %ld\n", quotient, by_448, whole);
  return 0;
}
