// fqa_quad_schedule.h — the order in which a wave of gemm_quad_kernel stages, reads and
// multiplies one tile's k steps, apart from what each operation does: the kernel runs it with
// the operations themselves, a host program with ones that record them and check that no LDS
// is read before it is filled or refilled before it is read.
#pragma once

#include "fqa_common.h"

namespace fqa {

// The tiles of gemm_quad_kernel: 4 waves, 2 x 2.  Each operand tile is two halves (rows
// 0 .. kBM/2 - 1 and the rest; W rows likewise) and a wave's kBM/2 x kBN/2 outputs are four
// quadrants, one per (x half, W half), of kQM x kQN 16 x 16 blocks.
template <int kBM_, int kBN_, int kRing_>
struct Quad {
  static constexpr int kBM = kBM_, kBN = kBN_, kRing = kRing_;
  static constexpr int kWM = 2, kWN = 2, kQM = kBM / 64, kQN = kBN / 64;
  static constexpr int kTM = 2 * kQM, kTN = 2 * kQN;
  static constexpr int kBK = 64, kPitch = 128;
  static constexpr int kHalfA = kBM / 2 * kPitch, kHalfB = kBN / 2 * kPitch;  // bytes per step
  static constexpr int kStage = 2 * (kHalfA + kHalfB);
  static constexpr int kWaves = 4, kThreads = 256;
  static constexpr int kDmaA = kBM / 64, kDmaB = kBN / 64;  // DMA instructions per wave per half
  static_assert(kRing >= 2 && kRing * kStage <= 160 * 1024, "LDS");
  __device__ static int swz(int r) { return (r >> 1) & 7; }
  typedef float4_t Block;
  static constexpr int kQuads = 1, kRowLanes = 16;
  __device__ static int row(int wm, int rb, int lane) {
    return (rb / kQM) * (kBM / 2) + wm * (kBM / 4) + (rb % kQM) * 16 + (lane & 15);
  }
  __device__ static int col(int wn, int cb, int, int lane) {
    return (cb / kQN) * (kBN / 2) + wn * (kBN / 4) + (cb % kQN) * 16 + 4 * (lane >> 4);
  }
};
using TileL = Quad<256, 256, 2>;
using TileP = Quad<192, 256, 2>;
using TileQ = Quad<256, 192, 2>;
using TileH = Quad<256, 128, 3>;
using TileM = Quad<128, 128, 5>;

// A step is 64 k of both operands, four halves (x rows: A0, A1; W rows: B0, B1), kRing steps
// in LDS, and four phases per wave, one per quadrant, in the order (A0,B0) (A0,B1) (A1,B1)
// (A1,B0).
//  * Every phase reads from LDS the half the next phase adds (B1, A1, A0(t+1), B0(t+1)), and
//    issues the DMA of one half (A1(t+R-1), A0(t+R), B0(t+R), B1(t+R), R = kRing), spread
//    between its MFMAs, so no wait sits in front of an MFMA and a half has 3 phases or more
//    to land.
//  * Two barriers per step, each behind a vmcnt that leaves the newest halves in flight:
//    after phase 2 A0(t+1) and B0(t+1) are in LDS for every wave, after phase 4 B1(t+1) and
//    A1(t+1).  A half's slot is refilled only after a barrier that follows every wave's last
//    use of it: fragments are consumed by MFMAs before the barrier, except A0(t+1)'s, which
//    the lgkmcnt before the second barrier waits for (B0(t+1)'s are newer; they are consumed
//    in phase 1 of t+1, a barrier before B0's refill).  read_first() ends the same way for
//    A0(0), which phase 2 of the first step refills.
//
// Ops has
//   stage_a(h, slot, i), stage_b(h, slot, i)   DMA instruction i of half h of the step that it
//                                              points at; stage_a1_prev: of the step before
//   keep(), advance(more)    "the step before" is now the one pointed at; point at the next
//   read_a(h, f), read_b(h, f)   fragment f = kk * blocks + block of half h
//   turn(d)                      reads are from d slots further on
//   mfma(i, j, r, c, kk)         x block r of half i, W block c of half j
//   wait_vm<N>(), wait_lgkm<N>(), barrier(), fence() (nothing moves across it)
template <class T>
struct QuadSchedule {
  static constexpr int kRing = T::kRing, kQM = T::kQM, kQN = T::kQN, dA = T::kDmaA, dB = T::kDmaB;
  int cur = 0;  // step t's slot
  int t = 0;

  // Steps 0 .. kRing - 1 on their way, but A1 of the last.
  template <class Ops>
  __host__ __device__ __forceinline__ void stage_first(Ops& o, int n) {
#pragma unroll
    for (int b = 0; b < kRing; ++b) {
#pragma unroll
      for (int i = 0; i < dA; ++i) o.stage_a(0, b, i);
#pragma unroll
      for (int i = 0; i < dB; ++i) o.stage_b(0, b, i);
#pragma unroll
      for (int i = 0; i < dB; ++i) o.stage_b(1, b, i);
      o.keep();
      if (b + 1 < kRing) {
#pragma unroll
        for (int i = 0; i < dA; ++i) o.stage_a(1, b, i);
        o.advance(b + 1 < n);
      }
    }
  }
  // Step 0 in LDS and its first fragments read.
  template <class Ops>
  __host__ __device__ __forceinline__ void read_first(Ops& o) {
    o.template wait_vm<2 * dB + dA + (kRing - 2) * 2 * (dA + dB)>();  // step 0
    o.barrier();
#pragma unroll
    for (int f = 0; f < 2 * kQM; ++f) o.read_a(0, f);
#pragma unroll
    for (int f = 0; f < 2 * kQN; ++f) o.read_b(0, f);
    o.template wait_lgkm<0>();  // (nothing keeps the compiler to this order of the reads)
    o.barrier();
  }

  // The steps of n from t up to `end`.
  template <class Ops>
  __host__ __device__ __forceinline__ void steps(Ops& o, int n, int end) {
    // One phase: the MFMAs of quadrant (x half i, W half j), kk outermost; between(q) places
    // fragment reads and DMA instructions after MFMA q.
    constexpr int kN = 2 * kQM * kQN;
    auto phase = [&](int i, int j, auto&& between) {
#pragma unroll
      for (int q = 0; q < kN; ++q) {
        o.mfma(i, j, q / kQN % kQM, q % kQN, q / (kQM * kQN));
        between(q);
        o.fence();
      }
    };
    // after MFMA q: those of `count` reads spread over the phase's first half, of `count` DMA
    // instructions spread over all of it
    auto reads = [&](int q, int count, auto&& f) {
#pragma unroll
      for (int e = 0; e < count; ++e)
        if (((2 * e + 1) * (kN / 2)) / (2 * count) == q) f(e);
    };
    auto stages = [&](int q, int count, auto&& f) {
#pragma unroll
      for (int e = 0; e < count; ++e)
        if (((2 * e + 1) * kN) / (2 * count) == q) f(e);
    };
    for (; t < end; ++t) {
      const int prev = cur == 0 ? kRing - 1 : cur - 1;
      const bool more = t + kRing < n;
      o.advance(more);
      phase(0, 0, [&](int q) {
        reads(q, 2 * kQN, [&](int f) { o.read_b(1, f); });
        stages(q, dA, [&](int i) { o.stage_a1_prev(prev, i); });  // A1(t + kRing - 1)
      });
      phase(0, 1, [&](int q) {
        reads(q, 2 * kQM, [&](int f) { o.read_a(1, f); });
        stages(q, dA, [&](int i) { o.stage_a(0, cur, i); });  // A0(t + kRing)
      });
      o.template wait_vm<dB + 2 * dA + (kRing - 2) * 2 * (dA + dB)>();  // A0(t+1), B0(t+1)
      o.barrier();
      o.turn(cur == kRing - 1 ? 1 - kRing : 1);  // to step t + 1's slot
      phase(1, 1, [&](int q) {
        reads(q, 2 * kQM, [&](int f) { o.read_a(0, f); });
        stages(q, dB, [&](int i) { o.stage_b(0, cur, i); });  // B0(t + kRing)
      });
      phase(1, 0, [&](int q) {  // B0(t+1)'s fragments as B0(t)'s are used up
        if (q >= kN / 2 && q < kN / 2 + kQN) o.read_b(0, q - kN / 2);
        if (q == kN - 1)
#pragma unroll
          for (int f = kQN; f < 2 * kQN; ++f) o.read_b(0, f);
        stages(q, dB, [&](int i) { o.stage_b(1, cur, i); });  // B1(t + kRing)
      });
      o.template wait_vm<2 * dB + dA + (kRing - 2) * 2 * (dA + dB)>();  // B1(t+1), A1(t+1)
      o.template wait_lgkm<2 * kQN>();  // A0(t+1) is read (B0's are newer)
      o.barrier();
      o.keep();
      cur = cur == kRing - 1 ? 0 : cur + 1;
    }
  }
};

}  // namespace fqa
