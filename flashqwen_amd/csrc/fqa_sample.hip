// fqa_sample.hip — token sampling over fp32 logits (gfx950).
//
// Replaces ArgmaxKernel + SampleKernel + LaunchSampleBatch (engine/src/kernels.cu:184-327):
// per row, greedy argmax when inv_temp <= 0, else temperature + top-p nucleus sampling
// with the caller's uniform draw u: weights w = exp((l - max) * inv_temp), the kept set
// is the fewest largest weights whose mass reaches top_p * sum(w), and the token is the
// first index at which the running kept mass reaches u * (kept mass).
//
// MI355X design: one 1024-thread workgroup per row.  Wave w owns a contiguous segment of
// the row and its lanes read 16 bytes each (1 KiB wave loads), so index order is (segment,
// step, lane, element) and the inverse-CDF pick keeps vocabulary order.  The reference finds
// the top-p threshold by 32 bisection passes over the row, each recomputing every weight;
// here it is a 3-level radix select on the weights' float bits (bits 30..20, 19..9, 8..0;
// positive floats order like their bit patterns), with exact integer mass histograms in LDS:
// the exact smallest kept weight after 3 levels, and with it each wave's kept mass.  A top-p
// row is read 3 times in full (max + sum, level 1, and a pass that copies the weights of the
// boundary bin into LDS, on which levels 2 and 3 run).  Only when the boundary bin may hold
// more than 16384 weights (copy_fits) is the row read a 4th time for level 3, and once more
// where the boundary lies below 2^-31 of the largest weight.  A temperature-only row is read
// once (its kept mass per wave is the rescaled pass-1 sum); the pick then reads 1/16 of one
// wave's segment.
//
// What bounds it: with a workgroup per row, what one CU loads and computes.  Each wave keeps a
// chunk of loads in flight while it works on the one before (4 KiB of them, 128 KiB per CU,
// where rows are few: 2 KiB with no overlap made a pass ~20 us however few the rows), and
// per-element work is kept free of branches and of atomics that meet: the running maximum is
// selected, not branched on, level 1 has a column per lane, room in the copy is taken once per
// chunk.  Sums keep one order (lane, step, element; then lanes; then waves) whatever the chunk,
// so a draw near a cumulative-mass boundary falls the same way.  151936 logits, 4 rows, before
// and after: greedy 21.6 -> 13.1 us, temperature 27.6 -> 18.6, top-p 0.9 79.2 -> 60.4, nearly flat rows
// 200.6 -> 74.8, masked rows (999 of 1000 at -inf) 51.7 -> 49.2; 256 rows (HBM and the caches
// carry the reads) 27.4 -> 25.6, 33.1 -> 29.0, 91.2 -> 82.0, 212.3 -> 100.8, 77.0 -> 76.8.
#include "fqa_common.h"
#include "fqa_sample_select.h"

#include <cfloat>

namespace fqa {
namespace {

constexpr int kSThreads = 1024;
constexpr int kSWaves = kSThreads / kWave;
constexpr int kBins = 2048;  // histogram bins per radix level (levels use 11, 11, 9 bits)

struct SampArgs {
  const float* logits;
  int vocab;
  long long stride;
  const float* inv_temp;
  const float* top_p;
  const float* u;
  int* out;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}
// Inclusive prefix sum over the wave's lanes.
__device__ __forceinline__ float wave_scan(float v) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const float x = __shfl_up(v, o, kWave);
    if (lane >= o) v += x;
  }
  return v;
}

// Descending scan of a mass histogram: the bin at which the mass of bins above it plus
// `above` first reaches `need` (need <= above + the histogram's total).  Returns the bin
// and, in *above_out, the mass above it.  Every thread takes 2 bins, highest first.
__device__ int find_crossing(const float* hist, int nbins, float above, float need,
                             float* sh, int* sres, float* sres_f, float* above_out) {
  const int t = threadIdx.x;
  const int b0 = nbins - 1 - 2 * t, b1 = b0 - 1;
  const float m0 = b0 >= 0 ? hist[b0] : 0.f, m1 = b1 >= 0 ? hist[b1] : 0.f;
  const float local = m0 + m1;
  // exclusive block scan of `local` in thread order (= descending bins)
  const int lane = t & (kWave - 1), w = t >> 6;
  const float incl = wave_scan(local);
  __syncthreads();
  if (lane == kWave - 1) sh[w] = incl;
  if (t == 0) {
    *sres = 0;  // lowest bin unless a crossing is found
    *sres_f = above;
  }
  __syncthreads();
  float before = above;
  for (int i = 0; i < w; ++i) before += sh[i];
  before += incl - local;
  if (before < need && before + local >= need) {
    if (b0 >= 0 && before + m0 >= need) {
      *sres = b0;
      *sres_f = before;
    } else {
      *sres = b1;
      *sres_f = before + m0;
    }
  }
  __syncthreads();
  *above_out = *sres_f;
  return *sres;
}

// Elements i .. i + 3 of the row (those past `end` as -inf: weight 0, never the largest).
__device__ __forceinline__ void load4(const float* lg, int i, int end, float (&x)[4]) {
  if (i + 3 < end) {
    __builtin_memcpy(x, lg + i, 16);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = i + e < end ? lg[i + e] : -INFINITY;
  }
}

// kChunk: 256-element steps whose loads a wave issues back to back and then works on (times:
// top-p 0.95, normal logits; masked: 999 of 1000 at -inf).
//  * 1 for rows of 16384 logits or less, which give a wave 4 steps at most, so that little of
//    a chunk lies past the row's end: 1000 / 4000 / 16000 logits 13.4 / 14.4 /
//    18.7 us against 15.5 / 17.8 / 18.5 with 4.
//  * 2 above 128 rows, where the caches carry the reads: 151936 logits, 200 / 256 rows 74.6 /
//    82.5 us against 76.8 / 87.9 with 4, 256 masked rows 76.5 against 80.4.
//  * 4 otherwise: 4 / 64 / 128 rows 60.8 / 66.1 / 68.7 us against 61.8 / 68.8 / 70.0 with 2.
template <int kChunk>
__global__ void __launch_bounds__(kSThreads) sample_kernel(SampArgs a) {
  typedef float Chunk[kChunk][4];
  __shared__ float sh[kSWaves];
  __shared__ float sh2[kSWaves];
  __shared__ int sres;
  __shared__ float sres_f;
  __shared__ int s_pick;

  const int row = blockIdx.x;
  const int N = a.vocab;
  const float* lg = a.logits + (long long)row * a.stride;
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  // Wave w of the row covers [seg0, seg1), a whole number of 256-element steps except at
  // the row's end; in a step lane l holds elements s0 + 4l .. s0 + 4l + 3.
  constexpr int kStep = 4 * kWave, kSpan = kChunk * kStep;
  const int seg = ((N + kSWaves * kStep - 1) / (kSWaves * kStep)) * kStep;
  const int seg0 = min(w * seg, N), seg1 = min(seg0 + seg, N);
  const float it = a.inv_temp[row];
  // f(chunk, its first index) for the segment's chunks of kChunk steps, in order; a chunk's
  // loads are issued before the chunk before it is used.
  auto load_chunk = [&](Chunk& x, int c0, int end) {
    if (c0 + kSpan <= end) {
#pragma unroll
      for (int u = 0; u < kChunk; ++u) __builtin_memcpy(x[u], lg + c0 + u * kStep + 4 * lane, 16);
      return;
    }
    // the chunk that the end cuts: no branches by lane, which would wait for one load before
    // the next
#pragma unroll
    for (int u = 0; u < kChunk; ++u) {
      const int s0 = c0 + u * kStep, i = s0 + 4 * lane;
      if (s0 + kStep <= end) {
        __builtin_memcpy(x[u], lg + i, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][e] = -INFINITY;
        if (s0 < end)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = lg[min(i + e, end - 1)];
            x[u][e] = i + e < end ? v : -INFINITY;
          }
      }
    }
  };
  auto for_chunks = [&](auto&& f) {
    if (seg0 >= seg1) return;
    Chunk x, next;
    load_chunk(x, seg0, seg1);
    for (int c0 = seg0; c0 < seg1; c0 += kSpan) {
      if (c0 + kSpan < seg1) load_chunk(next, c0 + kSpan, seg1);
      f(x, c0);
#pragma unroll
      for (int u = 0; u < kChunk; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][e] = next[u][e];
    }
  };
  auto chunk_max = [](const Chunk& x) {
    float m = x[0][0];
#pragma unroll
    for (int u = 0; u < kChunk; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) m = fmaxf(m, x[u][e]);
    return m;
  };

  if (it <= 0.f) {  // greedy: largest logit, the reference's tie order (greedy_key)
    float best = -INFINITY, wave_best = -INFINITY;  // this lane's, the wave's
    int bi = N;
    uint32_t bk = 0xffffffffu;
    for_chunks([&](const Chunk& x, int c0) {
      if (!__any(chunk_max(x) >= wave_best)) return;  // soon the usual case
#pragma unroll
      for (int u = 0; u < kChunk; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = c0 + u * kStep + 4 * lane + e;
          const uint32_t k = greedy_key(i);
          if (x[u][e] > best || (x[u][e] == best && k < bk)) {
            best = x[u][e];
            bi = i;
            bk = k;
          }
        }
      wave_best = wave_max(best);
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, kWave);
      const int oi = __shfl_xor(bi, o, kWave);
      const uint32_t ok = __shfl_xor(bk, o, kWave);
      if (ov > best || (ov == best && ok < bk)) {
        best = ov;
        bi = oi;
        bk = ok;
      }
    }
    __shared__ int wbi[kSWaves];
    __shared__ uint32_t wbk[kSWaves];
    if (lane == 0) {
      sh[w] = best;
      wbi[w] = bi;
      wbk[w] = bk;
    }
    __syncthreads();
    if (t == 0) {
      float b = sh[0];
      int i0 = wbi[0];
      uint32_t k0 = wbk[0];
      for (int k = 1; k < kSWaves; ++k)
        if (sh[k] > b || (sh[k] == b && wbk[k] < k0)) {
          b = sh[k];
          i0 = wbi[k];
          k0 = wbk[k];
        }
      a.out[row] = b > kGreedyFloor ? i0 : 0;  // nothing above -1e30 (all -inf/NaN): 0
    }
    return;
  }

  // pass 1: row max and total weight together (online: the running sum is rescaled when
  // the running max grows), merged across lanes and waves the same way.  The running max
  // starts at the lowest finite value, so a masked token (-inf) weighs 0 (exp2(-inf)).
  float lm = -FLT_MAX, ls = 0.f;
  for_chunks([&](const Chunk& x, int) {
#pragma unroll
    for (int u = 0; u < kChunk; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = x[u][e];
        const float w1 = __expf(-fabsf(v - lm) * it);  // of the smaller of the two
        ls = v > lm ? fmaf(ls, w1, 1.f) : ls + w1;
        lm = fmaxf(lm, v);
      }
  });
  auto merge = [&](float& m0, float& s0v, float m1, float s1) {
#pragma clang fp contract(off)
    const float mn = fmaxf(m0, m1);
    s0v = s0v * __expf((m0 - mn) * it) + s1 * __expf((m1 - mn) * it);
    m0 = mn;
  };
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) merge(lm, ls, __shfl_xor(lm, o, kWave), __shfl_xor(ls, o, kWave));
  if (lane == 0) {
    sh[w] = lm;
    sh2[w] = ls;
  }
  __syncthreads();
  float m = sh[0], Z = sh2[0];
  for (int k = 1; k < kSWaves; ++k) merge(m, Z, sh[k], sh2[k]);
  auto weight = [&](float v) { return __expf((v - m) * it); };

  // skm[w]: the kept mass of wave w's segment
  __shared__ float skm[kSWaves];
  // level 1 with a column per lane, then the copied boundary weights and a spare word per
  // lane, or level 3 per wave
  __shared__ unsigned long long big[kCols * kWave];
  __shared__ unsigned long long hcnt[kBins];
  __shared__ float hist[kBins];
  __shared__ unsigned long long s_kmc[kSWaves];
  __shared__ int s_ncand;
  static_assert((kCandCap + kWave) * 4 <= kCols * kWave * 8 && kSWaves * 512 <= kCols * kWave, "big");
  uint32_t thr = 0;  // kept: weights whose bits are >= thr (all, without top-p)
  const float tp = a.top_p[row];
  if (tp < 1.f) {
    // pass 2: level-1 histogram (weight bits 30..20).  Weights below
    // x_min = (1 - top_p) * Z / (2N) are left out: all of them together weigh less than
    // (1 - top_p) * Z / 2, so the top-p boundary lies above them.
    const float need = fmaxf(tp * Z, 1e-37f);  // top_p = 0 still keeps the largest weight
    const float x_min = 0.5f * (1.f - tp) * Z / (float)N;
    for (int b = t; b < kCols * kWave; b += kSThreads) big[b] = 0ull;
    for (int b = t; b < kBins; b += kSThreads) {
      hcnt[b] = 0ull;
      hist[b] = 0.f;
    }
    __syncthreads();
    for_chunks([&](const Chunk& x, int) {
#pragma unroll
      for (int u = 0; u < kChunk; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t bits = __float_as_uint(weight(x[u][e]));
          if (in_columns(bits, x_min))
            atomicAdd(&big[((bits >> 20) - kCol0) * kWave + lane], significand(bits));
        }
    });
    __syncthreads();
    {  // bin b's columns, 16 per thread
      const unsigned long long* src = big + t * 16;
      unsigned long long c = 0;
#pragma unroll
      for (int k = 0; k < 16; ++k) c += src[(k + t) & 15];
      c += __shfl_xor(c, 1, kWave);
      c += __shfl_xor(c, 2, kWave);
      if ((t & 3) == 0) {
        const int b = kCol0 + (t >> 2);
        hcnt[b] = c;
        hist[b] = bin_mass(c, b >> 3);
      }
    }
    __syncthreads();
    float above;
    int b1 = find_crossing(hist, kBins, 0.f, need, sh, &sres, &sres_f, &above);
    if (b1 < kCol0 && x_min < kBelowCols) {
      // the boundary lies further down (top_p within 2^-31 or so of 1, or rounding): the
      // bins below the columns too
      for_chunks([&](const Chunk& x, int) {
#pragma unroll
        for (int u = 0; u < kChunk; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t bits = __float_as_uint(weight(x[u][e]));
            const int b = (int)(bits >> 20);
            if (b < kCol0 && __uint_as_float(bits) >= x_min) atomicAdd(&hcnt[b], significand(bits));
          }
      });
      __syncthreads();
      for (int b = t; b < kBins; b += kSThreads) hist[b] = bin_mass(hcnt[b], b >> 3);
      __syncthreads();
      b1 = find_crossing(hist, kBins, 0.f, need, sh, &sres, &sres_f, &above);
    }
    const int e1 = b1 >> 3;  // the exponent field of every weight in bin b1
    // Bin 0 holds no counted weight: it means that there is no boundary (top_p so near to 1
    // that fp32 sums do not reach top_p * Z), and every weight is kept.
    const bool all = b1 == 0;
    const bool copy = all || copy_fits(hcnt[b1], b1, x_min);
    // pass 3: per lane, the mass of the weights above bin b1 (all kept), and the weights in
    // bin b1 copied into LDS (low 20 bits and the wave), on which level 2 (bits 19..9),
    // level 3 and the kept masses run without reading the row again; or level 2 here.
    uint32_t* cand = reinterpret_cast<uint32_t*>(big);
    __syncthreads();
    for (int b = t; b < kBins; b += kSThreads) hcnt[b] = 0ull;
    if (t == 0) s_ncand = 0;
    __syncthreads();
    float km1 = 0.f;
    for_chunks([&](const Chunk& x, int) {
      uint32_t bits[kChunk][4];
      int n = 0;
#pragma unroll
      for (int u = 0; u < kChunk; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float wv = weight(x[u][e]);
          bits[u][e] = __float_as_uint(wv);
          const int bb = (int)(bits[u][e] >> 20);
          km1 += bb > b1 ? wv : 0.f;
          n += bb == b1 ? 1 : 0;
        }
      if (all || !__any(n > 0)) return;
      if (copy) {
        // room for this lane's n weights: one addition per wave; then without branches,
        // what is not copied goes to a spare word
        const int incl = wave_incl_scan(n);
        int base = 0;
        if (lane == kWave - 1) base = atomicAdd(&s_ncand, incl);
        int slot = __builtin_amdgcn_readlane(base, kWave - 1) + incl - n;
#pragma unroll
        for (int u = 0; u < kChunk; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool in = (int)(bits[u][e] >> 20) == b1;
            cand[in ? slot : kCandCap + lane] = ((uint32_t)w << 20) | (bits[u][e] & 0xfffffu);
            slot += in ? 1 : 0;
          }
      } else {
#pragma unroll
        for (int u = 0; u < kChunk; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if ((int)(bits[u][e] >> 20) == b1)
              atomicAdd(&hcnt[(bits[u][e] >> 9) & 2047], significand(bits[u][e]));
      }
    });
    __syncthreads();
    const int nc = copy ? s_ncand : 0;
    if (copy) {
      for (int i = t; i < nc; i += kSThreads) {
        const uint32_t bits = ((uint32_t)b1 << 20) | (cand[i] & 0xfffffu);
        atomicAdd(&hcnt[(bits >> 9) & 2047], significand(bits));
      }
      __syncthreads();
    }
    for (int b = t; b < kBins; b += kSThreads) hist[b] = bin_mass(hcnt[b], e1);
    __syncthreads();
    const int b2 = find_crossing(hist, kBins, above, need, sh, &sres, &sres_f, &above);
    const uint32_t hi = ((uint32_t)b1 << 11) | (uint32_t)b2;
    if (copy) {
      // level 3 over the copied weights of (b1, b2), then each wave's kept mass: the
      // weights above bin b1 plus its copied weights at or above the threshold
      for (int b = t; b < 512; b += kSThreads) hcnt[b] = 0ull;
      if (t < kSWaves) s_kmc[t] = 0ull;
      __syncthreads();
      for (int i = t; i < nc; i += kSThreads) {
        const uint32_t bits = ((uint32_t)b1 << 20) | (cand[i] & 0xfffffu);
        if ((bits >> 9) == hi) atomicAdd(&hcnt[bits & 511], significand(bits));
      }
      __syncthreads();
      if (t < 512) hist[t] = bin_mass(hcnt[t], e1);
      __syncthreads();
      const int b3 = find_crossing(hist, 512, above, need, sh, &sres, &sres_f, &above);
      thr = (hi << 9) | (uint32_t)b3;
      for (int i = t; i < nc; i += kSThreads) {
        const uint32_t bits = ((uint32_t)b1 << 20) | (cand[i] & 0xfffffu);
        if (bits >= thr) atomicAdd(&s_kmc[cand[i] >> 20], significand(bits));
      }
      __syncthreads();
      const float km = wave_sum(km1);
      if (lane == 0) skm[w] = km + bin_mass(s_kmc[w], e1);
    } else {
      // pass 4: level 3 (bits 8..0 of the weights in (b1, b2)) as one histogram per
      // wave, and per wave the mass of the weights above (b1, b2), which are all kept:
      // the kept mass per wave then follows from the histograms without another pass
      for (int b = t; b < kSWaves * 512; b += kSThreads) big[b] = 0ull;
      __syncthreads();
      float km_hi = 0.f;
      for_chunks([&](const Chunk& x, int) {
#pragma unroll
        for (int u = 0; u < kChunk; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float wv = weight(x[u][e]);
            const uint32_t bits = __float_as_uint(wv);
            if ((bits >> 9) > hi) km_hi += wv;
            else if ((bits >> 9) == hi) atomicAdd(&big[w * 512 + (bits & 511)], significand(bits));
          }
      });
      __syncthreads();
      if (t < 512) {
        unsigned long long c = 0;
        for (int k = 0; k < kSWaves; ++k) c += big[k * 512 + t];
        hist[t] = bin_mass(c, e1);
      }
      __syncthreads();
      const int b3 = find_crossing(hist, 512, above, need, sh, &sres, &sres_f, &above);
      thr = (hi << 9) | (uint32_t)b3;
      unsigned long long c = 0;
      for (int b = b3 + lane; b < 512; b += kWave) c += big[w * 512 + b];
      float km = km_hi + bin_mass(c, e1);
      km = wave_sum(km);
      if (lane == 0) skm[w] = km;
    }
  } else {
    // every weight is kept: wave w's mass is its pass-1 sum rescaled to the row max
    if (t < kSWaves) skm[t] = sh2[t] * __expf((sh[t] - m) * it);
  }
  __syncthreads();

  // the pick: the wave whose kept mass [before, before + km) holds the draw u * total;
  // its segment is split into kSWaves sub-segments whose kept masses all waves sum at
  // once, and the wave owning the sub-segment that holds the draw walks it step by step
  // to the first kept token whose running mass reaches the draw
  auto kept = [&](float v) {
    const float wv = weight(v);
    return __float_as_uint(wv) >= thr ? wv : 0.f;
  };
  float total = 0.f;
  for (int k = 0; k < kSWaves; ++k) total += skm[k];
  const float target = a.u[row] * total;
  int ws = -1;
  float before = 0.f;
  {
    float acc = 0.f;
    for (int k = 0; k < kSWaves; ++k) {
      if (ws < 0 && acc <= target && target < acc + skm[k]) {
        ws = k;
        before = acc;
      }
      acc += skm[k];
    }
  }
  if (ws < 0) {  // a draw past the summed mass (rounding): the last token
    if (t == 0) a.out[row] = N - 1;
    return;
  }
  const int S0 = min(ws * seg, N), S1 = min(S0 + seg, N);
  const int sub = ((S1 - S0 + kSWaves * kStep - 1) / (kSWaves * kStep)) * kStep;
  const int u0 = min(S0 + w * sub, S1), u1 = min(u0 + sub, S1);
  // this wave's sub-segment; its first chunk stays in registers for the walk
  Chunk first_x;
  load_chunk(first_x, u0, u1);
  float m2 = 0.f;
  auto add_kept = [&](const Chunk& x) {
#pragma unroll
    for (int u = 0; u < kChunk; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) m2 += kept(x[u][e]);
  };
  add_kept(first_x);
  for (int c0 = u0 + kSpan; c0 < u1; c0 += kSpan) {
    Chunk x;
    load_chunk(x, c0, u1);
    add_kept(x);
  }
  m2 = wave_sum(m2);
  if (lane == 0) sh2[w] = m2;
  if (t == 0) s_pick = N - 1;
  __syncthreads();
  // the walker: the last sub-segment with kept mass that starts at or below the draw
  // (the first one with kept mass if rounding puts the draw below them all)
  int wk = -1, first = -1;
  float b2v = before, wb = before;
  for (int k = 0; k < kSWaves; ++k) {
    if (sh2[k] > 0.f) {
      if (first < 0) first = k;
      if (b2v <= target) {
        wk = k;
        wb = b2v;
      }
    }
    b2v += sh2[k];
  }
  if (wk < 0) {
    wk = first;
    wb = before;
  }
  if (w == wk) {
    float acc = wb;
    int last = -1;  // the last kept token walked so far
    for (int s0 = u0; s0 < u1; s0 += kStep) {
      const int i = s0 + 4 * lane;
      float x[4], kw[4];
      if (s0 - u0 < kSpan) {
        const int q = (s0 - u0) / kStep;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = first_x[0][e];
#pragma unroll
        for (int u = 1; u < kChunk; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = q == u ? first_x[u][e] : x[e];
      } else {
        load4(lg, i, u1, x);
      }
      float lsum = 0.f;
      int llast = -1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kw[e] = i + e < u1 ? kept(x[e]) : 0.f;
        lsum += kw[e];
        if (kw[e] > 0.f) llast = i + e;
      }
      const float incl = wave_scan(lsum);
      const float step = __shfl(incl, kWave - 1, kWave);
      // the first lane whose running mass reaches the draw, then its first such element
      const unsigned long long hit = __ballot(lsum > 0.f && acc + incl >= target);
      if (hit) {
        const int l = (int)__builtin_ctzll(hit);
        if (lane == l) {
          float run = acc + incl - lsum;
          // the first element whose running sum reaches the draw; if rounding leaves the
          // lane's own running sum short, its last kept element
          int pick = -1;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            run += kw[e];
            if (pick < 0 && kw[e] > 0.f && run >= target) pick = i + e;
          }
          s_pick = pick >= 0 ? pick : llast;
        }
        last = -2;
        break;
      }
      const unsigned long long has = __ballot(llast >= 0);
      if (has) last = __shfl(llast, 63 - __builtin_clzll(has), kWave);
      acc += step;
    }
    if (last >= 0 && lane == 0) s_pick = last;  // the draw lies past this sub-segment's sum
  }
  __syncthreads();
  if (t == 0) a.out[row] = s_pick;
}

}  // namespace
}  // namespace fqa

using namespace fqa;

extern "C" int fqa_sample(const float* logits, int32_t n_rows, int32_t vocab,
                          int64_t row_stride, const float* inv_temp, const float* top_p,
                          const float* u, int32_t* out, void* stream) {
  if (n_rows < 0 || vocab < 1 || vocab > (1 << 24) || row_stride < vocab) return FQA_EINVAL;
  if (n_rows == 0) return FQA_OK;
  if (!logits || !inv_temp || !top_p || !u || !out) return FQA_EINVAL;
  SampArgs a{logits, vocab, row_stride, inv_temp, top_p, u, out};
  const dim3 grid((unsigned)n_rows), block(kSThreads);
  const hipStream_t st = (hipStream_t)stream;
  if (vocab <= 16384)
    hipLaunchKernelGGL(sample_kernel<1>, grid, block, 0, st, a);
  else if (n_rows > 128)
    hipLaunchKernelGGL(sample_kernel<2>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(sample_kernel<4>, grid, block, 0, st, a);
  return hipGetLastError() == hipSuccess ? FQA_OK : FQA_ELAUNCH;
}
