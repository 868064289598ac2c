// any_quotient_check.cpp - the quotient of the register projection kernels over
// every binary32 input.
//
// tests/test_any_quotient.py writes any_quotient and quotient_class of
// projection_device.hpp, and class_quotient from the lines of kind_quotient that
// use them, into shipped.inc and builds this
// with g++ -O2 -mfma -ffp-contract=off -fopenmp, so what runs here is the
// kernels' own text.  Compared with div / s bit for bit for s = 1..4 (any NaN
// equals any NaN); s = 0 must give div * 0, since such a cell is not projected or
// adds a quotient made elsewhere.  The wavefronts at a wall give any_quotient
// constants instead of a class: both pairs, for s = 3 and 4.  Prints "<path>
// <mismatches>" for each; the exit status is 0 when all are 0.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#define __device__
#include "shipped.inc"

static float from_bits(uint32_t b) {
  float f;
  std::memcpy(&f, &b, 4);
  return f;
}
static bool same(float a, float b) {
  return (a != a && b != b) || std::memcmp(&a, &b, 4) == 0;
}

static long long g_step = 1;

template <class Want, class Got>
static int check(const char* path, const Want& want, const Got& got) {
  long long bad = 0;
#pragma omp parallel for reduction(+ : bad) schedule(static)
  for (long long k = 0; k < (1LL << 32); k += g_step) {
    const float div = from_bits((uint32_t)k);
    if (!same(want(div), got(div))) bad++;
  }
  std::printf("%s %lld\n", path, bad);
  return bad != 0;
}

int main(int argc, char** argv) {
  if (argc > 1) g_step = std::atoll(argv[1]);  // every step-th input only
  int fail = 0;
  for (int s = 0; s <= 4; s++) {
    volatile float divisor = (float)s;
    const float sf = divisor;  // not a constant: the division stays one
    const uint32_t c = quotient_class(s);
    char path[16];
    std::snprintf(path, sizeof path, "class %d:", s);
    fail |= check(path, [=](float d) { return s == 0 ? d * 0.0f : d / sf; },
                  [=](float d) { return class_quotient(d, c); });
  }
  volatile float three = 3.0f, four = 4.0f;
  const float s3 = three, s4 = four;
  fail |= check("wall 3:", [=](float d) { return d / s3; },
                [](float d) { return any_quotient(d, 1.0f / 3.0f, 3.0f); });
  fail |= check("wall 4:", [=](float d) { return d / s4; },
                [](float d) { return any_quotient(d, 0.25f, 4.0f); });
  return fail;
}
