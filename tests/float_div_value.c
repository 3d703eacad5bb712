/* Exhaustive check of the constant division of the flux5 / flux3 face values:
 * for every float x and the divisor d given on the command line, y = fma(e, r,
 * q) with q = RN(x r), e = fma(-q, d, x), r = RN(1/d) must equal RN(x / d)
 * (as values: a zero's sign may differ) unless y is NaN or subnormal (those
 * cases take a true division).  Prints the number of mismatches outside those
 * cases; exits 1 on any. */
#include <math.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static float D, R;
enum { NT = 8 };
typedef struct { uint64_t lo, hi, bad, fast; } Part;

static void* run(void* p) {
  Part* a = (Part*)p;
  for (uint64_t u = a->lo; u < a->hi; ++u) {
    uint32_t b = (uint32_t)u;
    float x;
    memcpy(&x, &b, 4);
    float q = x * R;
    float y = fmaf(fmaf(-q, D, x), R, q);
    int c = fpclassify(y);
    if (c == FP_SUBNORMAL || c == FP_NAN) continue;
    volatile float ref = x / D;
    a->fast++;
    if (!(y == ref)) a->bad++;
  }
  return 0;
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  D = (float)atof(argv[1]);
  R = 1.0f / D;
  Part P[NT];
  pthread_t t[NT];
  for (int i = 0; i < NT; ++i) {
    P[i].lo = (1ull << 32) * i / NT;
    P[i].hi = (1ull << 32) * (i + 1) / NT;
    P[i].bad = P[i].fast = 0;
    pthread_create(&t[i], 0, run, &P[i]);
  }
  uint64_t bad = 0, fast = 0;
  for (int i = 0; i < NT; ++i) {
    pthread_join(t[i], 0);
    bad += P[i].bad;
    fast += P[i].fast;
  }
  printf("d=%g fast-path inputs %llu mismatches %llu\n", D, (unsigned long long)fast, (unsigned long long)bad);
  return bad ? 1 : 0;
}
