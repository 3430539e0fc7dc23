// fqa_sample_select.h — what fqa_sample's radix select decides from its level-1 histogram,
// apart from the kernel so that a host program can run it too.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fqa {

// Histogram masses are exact integers: a weight with exponent field E adds its 24-bit
// significand, and a bin's mass is that sum times 2^(max(E, 1) - 150) (every bin holds one
// exponent).  ds_add_u64 runs at several times the rate of ds_add_f32 on gfx950, whose
// float adds were most of a top-p row's time; the sums also no longer depend on the order
// the atomics land in, so the kept set is the same on every run.
__host__ __device__ inline unsigned long long significand(uint32_t bits) {
  return (bits & 0x7fffffu) | (bits >= 0x800000u ? 0x800000u : 0u);
}
__host__ __device__ inline float bin_mass(unsigned long long sum, int exp_field) {
  return ldexpf((float)sum, (exp_field > 1 ? exp_field : 1) - 150);
}

constexpr int kCols = 256;  // level-1 bins with a column per lane: the 31 octaves below 1
constexpr int kCol0 = (127 << 3) + 8 - kCols;  // ... from this bin on (bits 30..20)
constexpr float kBelowCols = 0x1p-31f;  // weights below this lie below the columns
static_assert(kCol0 == (127 - 31) << 3, "kBelowCols");

// Whether a weight is counted in a column.  A NaN (of a NaN or infinite logit) has a bin past
// the columns, and compiled without NaN semantics the comparison with x_min may let it pass.
__host__ __device__ inline bool in_columns(uint32_t bits, float x_min) {
  return bits - ((uint32_t)kCol0 << 20) < ((uint32_t)kCols << 20) &&
         __builtin_bit_cast(float, bits) >= x_min;
}

constexpr int kCandCap = 16384;  // boundary-bin weights that the LDS copy holds

// Whether every weight in level-1 bin `bin` (bits 30..20) fits the LDS copy, `sum` being the
// bin's histogram: a normal weight's significand is 2^23 or more, so it holds at most sum >>
// 23 of them.  The histogram leaves weights below x_min out, so its sum says nothing of the
// bin that x_min cuts, nor of those below.  (In exact arithmetic the boundary lies at 2 x_min
// or above.  But Z is an fp32 sum, 2e-6 too large on some rows of 151936 logits and more on
// longer ones, and with 1 - top_p below that the bins above x_min need not reach top_p * Z.)
__host__ __device__ inline bool copy_fits(unsigned long long sum, int bin, float x_min) {
  return (bin >> 3) > 0 && bin > (int)(__builtin_bit_cast(uint32_t, x_min) >> 20) &&
         (sum >> 23) <= kCandCap;
}

}  // namespace fqa
