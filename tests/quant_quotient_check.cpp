// Host-side check of the FP8 quantization's quotient (quant_scale and
// quant_quotient of kvx_amd/csrc/fp_convert.h, the source the HIP kernels
// compile): wherever a scale is `fast`, the FP8 code of the quotient equals
// the code of the correctly rounded division.  Built and run by
// tests/test_quant_quotient.py; prints "<check> <mismatches> of <n>" lines.
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <random>
#include <vector>

#include "fp_convert.h"

using namespace kvx;

int main() {
  std::mt19937_64 rng(2024);
  long bad = 0, n = 0, fast = 0;
  auto check = [&](const QuantScale &q, float x) {
    const float a = quant_quotient(q, x);
    volatile float b = x / q.s;
    ++n;
    if (f32_to_e4m3(a) != f32_to_e4m3(b) || f32_to_e5m2(a) != f32_to_e5m2(b)) {
      if (bad++ < 5)
        fprintf(stderr, "x %08x s %08x: %08x vs %08x\n", f32_bits(x), f32_bits(q.s), f32_bits(a),
                f32_bits(b));
    }
  };
  // Boundaries between FP8 codes: midpoints of neighbours (and half the
  // smallest code), E4M3 first, then E5M2.
  std::vector<float> mids;
  for (int c = 0; c < 0x7E; ++c)
    mids.push_back((e4m3_to_f32((uint8_t)c) + e4m3_to_f32((uint8_t)(c + 1))) * 0.5f);
  for (int c = 0; c < 0x7B; ++c)
    mids.push_back((e5m2_to_f32((uint8_t)c) + e5m2_to_f32((uint8_t)(c + 1))) * 0.5f);
  mids.push_back(448.0f);
  mids.push_back(57344.0f);

  // Scales: significands at the edges of the fast rule (S mod 2^20 = 0 and
  // its neighbours at +-64), few-bit and all-ones ones, random ones, over
  // exponents that reach past both ends of the fast range.
  std::vector<uint32_t> scales;
  for (uint32_t top = 0; top < 8; ++top)
    for (int d : {0, 1, 17, 18, 19, 63, 64, 65, 66, 100, 0xFFF9D, 0xFFFBF, 0xFFFC0, 0xFFFC1,
                  0xFFFFF, 0x80000, 0x7FFFF, 0x80001})
      for (uint32_t e : {60u, 66u, 67u, 68u, 100u, 119u, 121u, 126u, 127u, 128u, 140u, 186u, 187u,
                         188u})
        scales.push_back((e << 23) | (top << 20) | (uint32_t)d);
  for (int i = 0; i < 4000; ++i)
    scales.push_back(((uint32_t)(60 + rng() % 130) << 23) | (uint32_t)(rng() & 0x7FFFFF));
  for (uint32_t u : scales) {
    for (uint32_t sign : {0u, 0x80000000u}) {
      const QuantScale q = quant_scale(bits_f32(u | sign));
      if (!q.fast) continue;
      ++fast;
      for (float m : mids) {
        // floats within 3 of the one nearest the boundary times the scale
        const uint32_t x = f32_bits(m * bits_f32(u));
        if (x < 4 || x >= 0x7F7FFFF0u) continue;
        for (int d = -3; d <= 3; ++d) check(q, bits_f32((x + d) | sign));
      }
      for (uint32_t x : {0u, 1u, 2u, 0x007FFFFFu, 0x00800000u, 0x7F7FFFFFu, 0x7F800000u,
                         0x7FC00000u})
        for (uint32_t xs : {0u, 0x80000000u}) check(q, bits_f32(x | xs));
      for (int i = 0; i < 200; ++i) check(q, bits_f32((uint32_t)rng()));
    }
  }
  printf("quotient %ld of %ld (%ld fast scales)\n", bad, n, fast);

  // What the rule leaves to the division: zeros, subnormals, infinities,
  // NaN, scales past 2^+-60 and those next to a multiple of 2^20.
  long wrong = 0;
  for (uint32_t u : {0u, 1u, 0x00800000u, 0x7F800000u, 0x7FC00000u, 0x217FFFFFu, 0x5D800001u,
                     0x3F800001u, 0x3F80003Fu, 0x3F8FFFFFu, 0x3F8FFFC1u})
    wrong += quant_scale(bits_f32(u)).fast || quant_scale(bits_f32(u | 0x80000000u)).fast;
  for (uint32_t u : {0x21800000u, 0x5D800000u, 0x3F800000u, 0x3F900000u, 0x3F800040u, 0x3F8FFFC0u})
    wrong += !quant_scale(bits_f32(u)).fast || !quant_scale(bits_f32(u | 0x80000000u)).fast;
  printf("rule %ld of 34\n", wrong);
  return 0;
}
