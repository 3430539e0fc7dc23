// sample_select.cpp — fqa_sample's level-1 select restated on the host (pass 1's fp32 sums in
// the kernel's order, the exact histogram of the weights from x_min on, the bin at which it
// reaches top_p * Z), with the kernel's own rule for the LDS copy of that bin's weights
// (copy_fits): wherever the rule says that they fit, all of them must, also those that the
// histogram left out.
//
//   sample_select VOCAB TOP_P... < logits    (VOCAB floats; inv_temp 1)
//
// prints one line per top_p: "bin x_min_bin counted in_bin fits", `counted` being the most
// weights that the bin's histogram allows for and `in_bin` what pass 3 copies.
//
//   sample_select columns
//
// checks that every weight counted in a column (in_columns) has one, whatever its bits.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "../../flashqwen_amd/csrc/fqa_sample_select.h"

using namespace fqa;

namespace {
constexpr int kWaves = 16, kLanes = 64, kBins = 2048;

uint32_t bits_of(float v) { return __builtin_bit_cast(uint32_t, v); }

void merge(float& m0, float& s0, float m1, float s1) {
  const float mn = std::max(m0, m1);
  const float a = s0 * expf(m0 - mn), b = s1 * expf(m1 - mn);
  s0 = a + b;
  m0 = mn;
}

// The row's maximum and total weight, summed as the kernel does: wave w's lane l takes
// elements 256 k + 4 l .. + 3 of the wave's segment, then lanes by xor, then waves.
void pass1(const std::vector<float>& x, float& m, float& Z) {
  const int N = (int)x.size(), step = 4 * kLanes;
  const int seg = ((N + kWaves * step - 1) / (kWaves * step)) * step;
  for (int w = 0; w < kWaves; ++w) {
    const int s0 = std::min(w * seg, N), s1 = std::min(s0 + seg, N);
    float lm[kLanes], ls[kLanes];
    for (int l = 0; l < kLanes; ++l) {
      lm[l] = -FLT_MAX;
      ls[l] = 0.f;
      for (int c = s0 + 4 * l; c < s1; c += step)
        for (int i = c; i < std::min(c + 4, s1); ++i) {
          const float w1 = expf(-fabsf(x[i] - lm[l]));
          ls[l] = x[i] > lm[l] ? fmaf(ls[l], w1, 1.f) : ls[l] + w1;
          lm[l] = std::max(lm[l], x[i]);
        }
    }
    for (int o = kLanes / 2; o > 0; o /= 2) {
      float m2[kLanes], s2[kLanes];
      for (int l = 0; l < kLanes; ++l) {
        m2[l] = lm[l];
        s2[l] = ls[l];
        merge(m2[l], s2[l], lm[l ^ o], ls[l ^ o]);
      }
      std::copy(m2, m2 + kLanes, lm);
      std::copy(s2, s2 + kLanes, ls);
    }
    if (w == 0) {
      m = lm[0];
      Z = ls[0];
    } else {
      merge(m, Z, lm[0], ls[0]);
    }
  }
}

int check_columns() {
  const uint32_t nan = 0x7fc00000u;
  for (float x_min : {0.f, 1e-9f, 0.5f, __builtin_bit_cast(float, nan)})
    for (uint32_t bin = 0; bin < 4096; ++bin)
      for (uint32_t low : {0u, 1u, 0xfffffu}) {
        const uint32_t bits = bin << 20 | low;
        const int col = (int)bin - kCol0;
        const bool in = in_columns(bits, x_min);
        if (in && (col < 0 || col >= kCols)) {
          std::printf("weight bits %08x, x_min %g: column %d\n", bits, x_min, col);
          return 1;
        }
        if (x_min == 0.f && in != (col >= 0 && col < kCols)) return 1;
      }
  return 0;
}
}  // namespace

int main(int argc, char** argv) {
  if (std::string(argv[1]) == "columns") return check_columns();
  const int N = std::atoi(argv[1]);
  std::vector<float> x(N);
  if (std::fread(x.data(), 4, N, stdin) != (size_t)N) return 2;
  float m, Z;
  pass1(x, m, Z);
  std::vector<uint32_t> wb(N);
  for (int i = 0; i < N; ++i) wb[i] = bits_of(expf(x[i] - m));
  for (int a = 2; a < argc; ++a) {
    const float tp = strtof(argv[a], nullptr);
    const float need = std::max(tp * Z, 1e-37f), x_min = 0.5f * (1.f - tp) * Z / (float)N;
    std::vector<unsigned long long> hist(kBins, 0);
    std::vector<long> in_bin(kBins, 0);
    for (uint32_t b : wb) {
      ++in_bin[b >> 20];
      if (__builtin_bit_cast(float, b) >= x_min) hist[b >> 20] += significand(b);
    }
    int b1 = 0;
    float above = 0.f;
    for (int b = kBins - 1; b >= 0; --b) {
      const float mass = bin_mass(hist[b], b >> 3);
      if (above < need && above + mass >= need) {
        b1 = b;
        break;
      }
      above += mass;
    }
    std::printf("%d %d %llu %ld %d\n", b1, (int)(bits_of(x_min) >> 20), hist[b1] >> 23, in_bin[b1],
                (int)copy_fits(hist[b1], b1, x_min));
  }
}
