// fqa_gemm.hip — the layer projections y = x · W^T on bf16 MFMA (gfx950).
//
// Replaces LaunchGemm (engine/src/kernels.cu:9-16: cublasGemmEx, bf16 in, fp32 compute,
// bf16 or fp32 out), which the step calls for QKV, o_proj, gate-up, down and lm_head
// (engine/src/model_runtime.cu:261, 280, 285, 288, 322).  x is [M, K] and W is [N, K],
// both K-contiguous (the reference's weight layout), y is [M, N].
//
// MI355X design:
//  * Four kernels, chosen by a model of their times (gemm_plan):
//    - gemm_quad_kernel: tiles of 128 to 256 rows and columns on 4 waves, one per SIMD;
//    - gemm_slab_kernel: up to 96 x 64 outputs per workgroup for few rows, its waves dividing K
//      and summing in LDS, so that decode steps fill the CUs without a second kernel;
//    - gemm_kernel: 32 and 64 rows by 128 columns where W is wide enough to fill the CUs;
//    - where the tiles alone still leave CUs idle, K is split over workgroups that leave fp32
//      partials, which gemm_reduce_kernel sums (or fqa_qkv_proj_append's append kernel reads).
//  * Both operands move global -> LDS by DMA (global_load_lds_dwordx4, 1 KiB per wave
//    instruction: 8 rows x 128 bytes) into a ring of k steps, as deep as 160 KiB of LDS
//    allows, every slot in flight.  A DMA lane's 16 bytes land at LDS byte 16 * lane, so the
//    bank swizzle (swz) is applied on the global side of the DMA.
//  * Workgroups are dealt to the 8 XCDs round robin; tile_of() renumbers them so that the
//    workgroups on one XCD walk 8 m tiles per n tile and share W and x tiles in its L2.

#include "fqa_append_math.h"
#include "fqa_common.h"
#include "fqa_gemm_internal.h"
#include "fqa_quad_schedule.h"

#include <type_traits>

namespace fqa {
namespace {

constexpr int kGK = 64;  // K granularity of the shapes accepted (k steps are 32 or 64)

// Tile shapes.  kWM x kWN waves; a wave owns kTM x kTN blocks of 32 x 32 outputs; K
// advances kBK (32 or 64) per step, through a ring of kRing steps in LDS (kRing - 1 in
// flight ahead of the MFMAs).  An LDS row of a step holds kBK bf16 (kPitch bytes) in
// 16-byte chunks, chunk c of row r at c ^ swz(r): (r >> 1) & 7 for 8 chunks, (r >> 2) & 3
// for 4.  A ds_read_b128 is served 16 lanes at a time from the 64 banks (256 bytes); the
// 16 lanes of a fragment read take one chunk of 16 consecutive rows, and with this swizzle
// those land on 16 distinct 16-byte bank groups.
template <int kWM_, int kWN_, int kTM_, int kTN_, int kRing_, int kBK_ = 64>
struct Tile {
  static constexpr int kWM = kWM_, kWN = kWN_, kTM = kTM_, kTN = kTN_, kRing = kRing_;
  static constexpr int kBK = kBK_, kPitch = kBK * 2, kChunks = kBK / 8, kKK = kBK / 16;
  static constexpr int kRowsPerDma = 1024 / kPitch;
  static constexpr int kBM = kWM * kTM * 32, kBN = kWN * kTN * 32;
  static constexpr int kABytes = kBM * kPitch, kBBytes = kBN * kPitch;
  static constexpr int kStage = kABytes + kBBytes;
  static constexpr int kWaves = kWM * kWN, kThreads = 64 * kWaves;
  // DMA instructions per wave per step
  static constexpr int kDmaA = kBM / kRowsPerDma / kWaves, kDmaB = kBN / kRowsPerDma / kWaves;
  static_assert(kBK == 32 || kBK == 64, "k step");
  static_assert(kWaves == 4 || kWaves == 8, "4 or 8 waves");
  static_assert(kDmaA * kRowsPerDma * kWaves == kBM && kDmaB * kRowsPerDma * kWaves == kBN,
                "DMA split");
  static_assert(kRing * kStage <= 160 * 1024, "LDS");
  static_assert((kRing - 1) * (kDmaA + kDmaB) < 64, "vmcnt");
  __device__ static int swz(int r) { return kChunks == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3); }
  // Accumulator block (rb, cb) of wave (wm, wn): the MFMAs compute the transposed block (W
  // fragments as the row operand), so a lane holds one row of the tile and kQuads runs of 4
  // consecutive columns.
  typedef float16_t Block;
  static constexpr int kQuads = 4, kRowLanes = 32;
  __device__ static int row(int wm, int rb, int lane) { return (wm * kTM + rb) * 32 + (lane & 31); }
  __device__ static int col(int wn, int cb, int q, int lane) {
    return (wn * kTN + cb) * 32 + 8 * q + 4 * (lane >> 5);
  }
};
template <class T>
constexpr bool kIsQuad = false;
template <int M, int N, int R>
constexpr bool kIsQuad<Quad<M, N, R>> = true;
using TileS = Tile<1, 4, 2, 1, 6>;  // 64 x 128
using TileT = Tile<1, 4, 1, 1, 8>;  // 32 x 128: a few decode rows

struct GemmArgs {
  const uint16_t* x;
  const uint16_t* w;
  void* y;
  float* part;  // [splits][M][N] fp32 when splits > 1
  long long ldx, ldw, ldy;
  int M, N, K;
  int splits;
  int m_tiles, n_tiles;
  float* amax_v;  // argmax mode: per (row, n tile) the tile's largest value and its column
  int* amax_i;
  GemmAppend app;  // append mode: y is the qkv buffer (row stride ldy)
};

__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile(
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(off), "s"(base), "{m0}"(lds)
      : "memory");
}
// ... of W, with the non-temporal hint (kNT) where no other workgroup reads it: 1.2 GB
// streamed by 256 workgroups 198 -> 176 us, 201 MB 41 -> 37.5 us (DMA alone); gate_up at 6
// rows 42.8 -> 39.0 us.  With K split over workgroups it costs instead (6144 x 4096 at 64
// rows 17.8 -> 19.3 us).
template <bool kNT>
__device__ __forceinline__ void dma16_w(const void* base, uint32_t off, uint32_t lds) {
  if constexpr (kNT)
    asm volatile(
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %1 nt"
        :
        : "v"(off), "s"(base), "{m0}"(lds)
        : "memory");
  else
    dma16(base, off, lds);
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// Wait until at most n * kPer of this wave's loads are outstanding, n in [0, kMax].
template <int kPer, int kMax>
__device__ __forceinline__ void wait_steps(int n) {
  if constexpr (kMax <= 0) {
    wait_vm<0>();
  } else {
    if (n >= kMax)
      wait_vm<kMax * kPer>();
    else
      wait_steps<kPer, kMax - 1>(n);
  }
}
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// Workgroup -> (m tile, n tile, split).  Workgroups are dealt to the 8 XCDs round robin,
// so the linear id is first turned into an index that runs contiguously within an XCD;
// that index walks the tiles in groups of 8 m tiles per n tile (consecutive workgroups on
// an XCD share a W tile, and 4 consecutive n tiles share the group's x tiles in L2).
__device__ __forceinline__ void tile_of(const GemmArgs& a, int& tm, int& tn, int& sp) {
  const int G = a.m_tiles * a.n_tiles * a.splits;
  const int L = blockIdx.x;
  int t = L;
  if ((G & 7) == 0) t = (L & 7) * (G >> 3) + (L >> 3);
  const int per = a.m_tiles * a.n_tiles;
  sp = t / per;
  t -= sp * per;
  constexpr int kGroup = 8;
  const int span = kGroup * a.n_tiles;
  const int g = t / span, m0 = g * kGroup;
  const int gs = min(a.m_tiles - m0, kGroup);
  const int r = t - g * span;
  tm = m0 + r % gs;
  tn = r / gs;
}

// Append mode: the bf16 output tile is staged in LDS with this row pitch (16 bytes of
// padding rotate consecutive rows across the banks).
template <class T>
constexpr int kTilePitch = T::kBN * 2 + 16;
// ... followed by the tile rows' positions and slots (int32 each)
template <class T>
constexpr int kAppendLds = T::kBM * kTilePitch<T> + T::kBM * 8;
template <class T, bool kAppend>
constexpr int kGemmLds = (kAppend || kIsQuad<T>) && kAppendLds<T> > T::kRing * T::kStage
                             ? kAppendLds<T>
                             : T::kRing * T::kStage;

// The tile rounded to bf16 in LDS, row r at r * kTilePitch (every wave's reads of the operand
// ring are done first; on return every wave sees the tile).
template <class T>
__device__ __forceinline__ void stage_tile(char* lds, const typename T::Block (&acc)[T::kTM][T::kTN],
                                           int wm, int wn, int lane) {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's reads of the ring are done
  barrier();                           // ... and every wave's: the LDS is free
#pragma unroll
  for (int rb = 0; rb < T::kTM; ++rb)
#pragma unroll
    for (int cb = 0; cb < T::kTN; ++cb)
#pragma unroll
      for (int q = 0; q < T::kQuads; ++q)
        *reinterpret_cast<uint2*>(lds + T::row(wm, rb, lane) * kTilePitch<T> +
                                  T::col(wn, cb, q, lane) * 2) =
            make_uint2(pack_bf16x2(acc[rb][cb][4 * q], acc[rb][cb][4 * q + 1]),
                       pack_bf16x2(acc[rb][cb][4 * q + 2], acc[rb][cb][4 * q + 3]));
  __builtin_amdgcn_s_waitcnt(0xC07F);
  barrier();
}

template <class T>
__device__ void append_epilogue(const GemmArgs& a, char* lds, const typename T::Block (&acc)[T::kTM][T::kTN],
                                int row0, int col0, int wm, int wn, int w, int lane);

// K in four segments, begun at another one by workgroups that run side by side: in lockstep
// at one k offset of rows a power of two apart they meet on the same HBM channels (DMA alone:
// 201 MB by 256 workgroups 37.7 -> 31.3 us, by 192 40.4 -> 30.2; 67 MB 17.9 -> 11.8).  The
// sums stay independent of where a workgroup begins, so equal columns give equal values: the
// segments' sums a0..a3, in the order taken, add up as (a0 + a2) + (a1 + a3), which any
// rotation leaves the same.
struct Segments {
  int n, start;  // steps, the first segment
  __device__ int first() const { return start * n / 4; }  // its first step
  __device__ int end(int taken) const {  // steps of the segments 0 .. taken, in the order taken
    const int e = start + taken + 1;
    return (e > 4 ? (e - 4) * n / 4 + n : e * n / 4) - first();
  }
};
// Segment e (0..3 in the order taken) is complete in acc: kept in (or added to) sum[e & 1],
// acc cleared for the next; after the last, acc is the total.
template <int e, class B, int kM, int kN>
__device__ __forceinline__ void close_segment(B (&sum)[2][kM][kN], B (&acc)[kM][kN]) {
#pragma unroll
  for (int rb = 0; rb < kM; ++rb)
#pragma unroll
    for (int cb = 0; cb < kN; ++cb) {
      if constexpr (e < 2)
        sum[e][rb][cb] = acc[rb][cb];
      else if constexpr (e == 2)
        sum[0][rb][cb] += acc[rb][cb];
      else
        acc[rb][cb] = sum[0][rb][cb] + (sum[1][rb][cb] + acc[rb][cb]);
      if constexpr (e < 3)
#pragma unroll
        for (int i = 0; i < (int)(sizeof(B) / 4); ++i) acc[rb][cb][i] = 0.f;
    }
}
// steps(end) runs the steps up to `end`.
template <class F, class B, int kM, int kN>
__device__ __forceinline__ void run_segments(const Segments& segs, B (&acc)[kM][kN], F&& steps) {
  B sum[2][kM][kN];
  steps(segs.end(0));
  close_segment<0>(sum, acc);
  steps(segs.end(1));
  close_segment<1>(sum, acc);
  steps(segs.end(2));
  close_segment<2>(sum, acc);
  steps(segs.n);
  close_segment<3>(sum, acc);
}

// What a workgroup does with its tile's accumulators.
template <class T, bool kF32Out, bool kPartial, bool kArgmax, bool kAppend>
__device__ __forceinline__ void tile_epilogue(const GemmArgs& a, char* lds,
                                              const typename T::Block (&acc)[T::kTM][T::kTN], int row0,
                                              int col0, int tn, int sp, int wm, int wn, int w,
                                              int lane) {
  if constexpr (kAppend) {
    append_epilogue<T>(a, lds, acc, row0, col0, wm, wn, w, lane);
    return;
  }
  if constexpr (kArgmax) {
    // per row of the tile: the largest value and its column (ties in the reference's greedy
    // order, greedy_key), over this lane's values, then the wave's other lanes of the same
    // row, then the tile's kWN column waves through LDS (free once every wave's reads are
    // done)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    barrier();
    float* sv = reinterpret_cast<float*>(lds);
    int* si = reinterpret_cast<int*>(lds + T::kBM * T::kWN * 4);
#pragma unroll
    for (int rb = 0; rb < T::kTM; ++rb) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
      uint32_t bk = 0xffffffffu;
#pragma unroll
      for (int cb = 0; cb < T::kTN; ++cb)
#pragma unroll
        for (int q = 0; q < T::kQuads; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = acc[rb][cb][4 * q + e];
            const int n = col0 + T::col(wn, cb, q, lane) + e;
            const uint32_t k = greedy_key(n);
            if (v > bv || (v == bv && k < bk)) {
              bv = v;
              bi = n;
              bk = k;
            }
          }
#pragma unroll
      for (int o = T::kRowLanes; o < kWave; o *= 2) {
        const float ov = __shfl_xor(bv, o, kWave);
        const int oi = __shfl_xor(bi, o, kWave);
        if (ov > bv || (ov == bv && greedy_key(oi) < greedy_key(bi))) {
          bv = ov;
          bi = oi;
        }
      }
      const int r = T::row(wm, rb, lane);  // row within the tile
      if (lane < T::kRowLanes) {
        sv[r * T::kWN + wn] = bv;
        si[r * T::kWN + wn] = bi;
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    barrier();
    for (int r = threadIdx.x; r < T::kBM; r += T::kThreads) {
      const int m = row0 + r;
      if (m >= a.M) continue;
      float bv = sv[r * T::kWN];
      int bi = si[r * T::kWN];
      for (int k = 1; k < T::kWN; ++k)
        if (sv[r * T::kWN + k] > bv ||
            (sv[r * T::kWN + k] == bv && greedy_key(si[r * T::kWN + k]) < greedy_key(bi))) {
          bv = sv[r * T::kWN + k];
          bi = si[r * T::kWN + k];
        }
      // row-major by row, so the reduction reads each row's maxima contiguously (these
      // scattered 4-byte stores are a few hundred per tile of a long kernel)
      a.amax_v[(long long)m * a.n_tiles + tn] = bv;
      a.amax_i[(long long)m * a.n_tiles + tn] = bi;
    }
    return;
  }

  if constexpr (kIsQuad<T> && !kPartial && !kF32Out) {
    // Stored straight from the accumulators, every instruction touches 16 rows with 32 bytes
    // each, ~4 address cycles per row (7 us per tile); the tile goes through LDS instead and
    // out as whole rows of the tile.
    stage_tile<T>(lds, acc, wm, wn, lane);
    uint16_t* y = static_cast<uint16_t*>(a.y) + col0;
    const bool wide = (a.ldy & 7) == 0;  // rows start on 16 bytes
    constexpr int kRowChunks = T::kBN / 8, kRows = kWave / kRowChunks;  // rows per store
    for (int r0 = kRows * w; r0 < T::kBM; r0 += kRows * T::kWaves) {
      const int r = r0 + lane / kRowChunks, c = lane % kRowChunks, m = row0 + r;
      if (lane >= kRows * kRowChunks) break;  // 192 columns: 2 rows on 48 lanes
      const uint4 v = *reinterpret_cast<const uint4*>(lds + r * kTilePitch<T> + c * 16);
      if (m >= a.M) continue;
      uint16_t* d = y + m * a.ldy + c * 8;
      if (wide) {
        *reinterpret_cast<uint4*>(d) = v;
      } else {
        *reinterpret_cast<uint2*>(d) = make_uint2(v.x, v.y);
        *reinterpret_cast<uint2*>(d + 4) = make_uint2(v.z, v.w);
      }
    }
    return;
  }
  // one 16-byte (fp32) or 8-byte (bf16) store per run of 4 columns
#pragma unroll
  for (int rb = 0; rb < T::kTM; ++rb) {
    const int m = row0 + T::row(wm, rb, lane);
    if (m >= a.M) continue;
#pragma unroll
    for (int cb = 0; cb < T::kTN; ++cb)
#pragma unroll
      for (int q = 0; q < T::kQuads; ++q) {
        const int n = col0 + T::col(wn, cb, q, lane);
        const float4 v = make_float4(acc[rb][cb][4 * q], acc[rb][cb][4 * q + 1],
                                     acc[rb][cb][4 * q + 2], acc[rb][cb][4 * q + 3]);
        if (kPartial)
          *reinterpret_cast<float4*>(a.part + ((long long)sp * a.M + m) * a.N + n) = v;
        else if (kF32Out)
          *reinterpret_cast<float4*>(static_cast<float*>(a.y) + m * a.ldy + n) = v;
        else
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.y) + m * a.ldy + n) =
              make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
      }
  }
}

// The tiles of 32 and 64 rows, which stream W once (one row tile, no K split): gate_up at 6 /
// 64 rows 45.5 / 47.5 -> 32.8 / 38.3 us with the segments and the non-temporal W loads,
// lm_head at 2 rows 264 -> 193 us (6.5 TB/s).
template <class T, bool kF32Out, bool kArgmax = false>
__global__ void __launch_bounds__(T::kThreads, 1) gemm_kernel(GemmArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[kGemmLds<T, false>];
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w % T::kWM, wn = w / T::kWM;
  int tm, tn, sp;
  tile_of(a, tm, tn, sp);
  const int row0 = tm * T::kBM, col0 = tn * T::kBN;
  const int n_my = a.K / T::kBK;
  const uint16_t* xk = a.x;
  const uint16_t* wk = a.w;

  // DMA sources: wave w's instruction i covers rows kRowsPerDma (w kDmaA + i) + lane /
  // kChunks of the x tile (likewise of the W tile); lane fills LDS chunk lane % kChunks
  // of its row, so it reads global chunk (lane % kChunks) ^ swz(row)
  const int drow = lane / T::kChunks, dlc = lane % T::kChunks;
  uint32_t off_a[T::kDmaA], off_b[T::kDmaB];
#pragma unroll
  for (int i = 0; i < T::kDmaA; ++i) {
    const int tr = T::kRowsPerDma * (w * T::kDmaA + i) + drow;  // row within the tile
    const int r = min(row0 + tr, a.M - 1);
    off_a[i] = (uint32_t)((long long)r * a.ldx * 2) + (dlc ^ T::swz(tr)) * 16;
  }
#pragma unroll
  for (int i = 0; i < T::kDmaB; ++i) {
    const int tr = T::kRowsPerDma * (w * T::kDmaB + i) + drow;
    off_b[i] = (uint32_t)((long long)(col0 + tr) * a.ldw * 2) + (dlc ^ T::swz(tr)) * 16;
  }
  // load q (0 .. kDmaA + kDmaB - 1) of this wave's share of the workgroup's j-th k step
  const Segments segs{n_my, (int)(blockIdx.x >> 3) & 3};
  const int rot = segs.first();
  auto issue_one = [&](int j, int q) {
    const uint32_t dst = lds_base + (j % T::kRing) * T::kStage;
    j += rot;
    if (j >= n_my) j -= n_my;
    if (q < T::kDmaA)
      dma16(xk + (long long)j * T::kBK, off_a[q], dst + (w * T::kDmaA + q) * 1024);
    else
      dma16_w<true>(wk + (long long)j * T::kBK, off_b[q - T::kDmaA],
                     dst + T::kABytes + (w * T::kDmaB + q - T::kDmaA) * 1024);
  };
  auto issue = [&](int j) {
#pragma unroll
    for (int q = 0; q < T::kDmaA + T::kDmaB; ++q) issue_one(j, q);
  };

  // fragment reads: lane reads row (lane & 31) of a 32-row block, k chunk 2 kk + lane/32,
  // stored at chunk (2 kk + lane/32) ^ swz(lane & 31)
  const int a_off = (wm * T::kTM * 32 + (lane & 31)) * T::kPitch;
  const int b_off = T::kABytes + (wn * T::kTN * 32 + (lane & 31)) * T::kPitch;
  int phk[T::kKK];
#pragma unroll
  for (int kk = 0; kk < T::kKK; ++kk) phk[kk] = ((2 * kk + (lane >> 5)) ^ T::swz(lane & 31)) * 16;

  float16_t acc[T::kTM][T::kTN];
#pragma unroll
  for (int rb = 0; rb < T::kTM; ++rb)
#pragma unroll
    for (int cb = 0; cb < T::kTN; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rb][cb][i] = 0.f;

  // Pipeline: every ring slot holds a step in flight.  The one barrier per step sits
  // before the step's last MFMAs: by then every wave has read all of the step's
  // fragments, so its slot is refilled (step s + kRing) and the next step's first
  // fragments are read while those MFMAs run.
  bf16x8 af[2][T::kTM], bfg[2][T::kTN];
  auto read_frags = [&](int buf, int s, int kk) {
    const char* sb = lds + (s % T::kRing) * T::kStage;
#pragma unroll
    for (int rb = 0; rb < T::kTM; ++rb)
      af[buf][rb] = *reinterpret_cast<const bf16x8*>(sb + a_off + rb * 32 * T::kPitch + phk[kk]);
#pragma unroll
    for (int cb = 0; cb < T::kTN; ++cb)
      bfg[buf][cb] = *reinterpret_cast<const bf16x8*>(sb + b_off + cb * 32 * T::kPitch + phk[kk]);
  };
  constexpr int kPer = T::kDmaA + T::kDmaB;
#pragma unroll
  for (int j = 0; j < T::kRing; ++j)
    if (j < n_my) issue(j);
  wait_steps<kPer, T::kRing - 1>(min(T::kRing - 1, n_my - 1));
  barrier();  // step 0 landed for every wave
  read_frags(0, 0, 0);
  int s = 0;
  auto steps = [&](int end) {
    for (; s < end; ++s) {
#pragma unroll
      for (int kk = 0; kk < T::kKK; ++kk) {
        if (kk + 1 < T::kKK) {
          read_frags((kk + 1) & 1, s, kk + 1);
        } else if (s + 1 < n_my) {
          // step s + 1 landed (steps up to s + kRing - 1 may still be in flight)
          wait_steps<kPer, T::kRing - 2>(min(T::kRing - 2, n_my - 2 - s));
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of step s done
          barrier();
          read_frags(0, s + 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep those reads ahead of this sub-step's MFMAs
        // On the last sub-step the freed slot's refill (step s + kRing) is issued one load
        // after each MFMA, so the wave's load issue overlaps its own MFMAs.
        const bool refill = kk + 1 == T::kKK && s + T::kRing < n_my;
        constexpr int kMfma = T::kTM * T::kTN;
#pragma unroll
        for (int q = 0; q < (kMfma > kPer ? kMfma : kPer); ++q) {
          if (q < kMfma) {
            const int rb = q / T::kTN, cb = q % T::kTN;
            acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfg[kk & 1][cb], af[kk & 1][rb],
                                                                  acc[rb][cb], 0, 0, 0);
          }
          if (q < kPer && refill) issue_one(s + T::kRing, q);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  run_segments(segs, acc, steps);

  tile_epilogue<T, kF32Out, false, kArgmax, false>(a, lds, acc, row0, col0, tn, sp, wm, wn, w, lane);
}

// The large tiles: one wave per SIMD, each a quarter of the tile (128 x 128 of 256 x 256), its
// steps in the order of QuadSchedule.
//  * What bounds the 256 x 256 tile: the MFMAs at the clock the card holds under them (taking
//    all DMA out of the loop changes 289 us to 292 on 8192 x 6144 x 4096, all waits and
//    barriers to 282), then ~5 us per tile to start and to store.  16 x 16 x 32 MFMAs beat
//    32 x 32 x 16 here (289 against 313 us): 16-cycle steps leave the wave's other
//    instructions more places to issue.  128 x 128 per wave reads each fragment for 8 MFMAs.
//  * 256 x 256, 8192 rows, qkv / o_proj / gate_up / down: 325 / 221 / 1285 / 604 us (8 waves,
//    32 x 32 MFMAs, the next step staged in one burst) -> 284 / 192 / 1158 / 545 us,
//    1.42-1.51 PFLOP/s.  256 x 128 and 128 x 128 against their 8- and 4-wave predecessors:
//    qkv at 1000 rows 61 -> 52 us, o_proj at 700 rows 39 -> 33, gate_up at 512 rows (256 x
//    256) 122 -> 94, down at 700 rows (256 x 256, K split 5 ways) 93 -> 74.
// QuadSchedule's operations, for one wave.  LDS: the x halves of slot b at b * 2 kHalfA, the
// W halves at kB + b * 2 kHalfB.
template <class T, bool kNT>
struct QuadOps {
  static constexpr int kQM = T::kQM, kQN = T::kQN, kB = T::kRing * 2 * T::kHalfA;
  char* lds;
  uint32_t dst_a, dst_b;  // this wave's share of a half, in slot 0
  uint32_t off_a[2][T::kDmaA], off_b[2][T::kDmaB];
  // where the newest staged step starts (past the end the last step is staged again, never
  // read, so that every wait count holds), and the x of the step before it
  const uint16_t *xs, *ws, *xs_prev;
  int n, pos;  // steps; the one that xs and ws point at
  long long kstride;
  int pa[2], pb[2];
  bf16x8 af[2][kQM][2], bf[2][kQN][2];  // [half][r][kk]
  float4_t acc[T::kTM][T::kTN];

  __device__ __forceinline__ void stage_a(int h, int slot, int i) {
    dma16(xs, off_a[h][i], dst_a + (2 * slot + h) * T::kHalfA + i * 1024);
  }
  __device__ __forceinline__ void stage_a1_prev(int slot, int i) {
    dma16(xs_prev, off_a[1][i], dst_a + (2 * slot + 1) * T::kHalfA + i * 1024);
  }
  __device__ __forceinline__ void stage_b(int h, int slot, int i) {
    dma16_w<kNT>(ws, off_b[h][i], dst_b + (2 * slot + h) * T::kHalfB + i * 1024);
  }
  __device__ __forceinline__ void keep() { xs_prev = xs; }
  __device__ __forceinline__ void advance(bool more) {
    if (!more) return;
    const long long d = ++pos == n ? kstride - n * kstride : kstride;
    pos = pos == n ? 0 : pos;
    xs += d;
    ws += d;
  }
  // fragment f = kk * (blocks) + r of half h, in the slot that pa / pb point at
  __device__ __forceinline__ void read_a(int h, int f) {
    af[h][f % kQM][f / kQM] = *reinterpret_cast<const bf16x8*>(
        lds + pa[f / kQM] + h * T::kHalfA + (f % kQM) * 16 * T::kPitch);
  }
  __device__ __forceinline__ void read_b(int h, int f) {
    bf[h][f % kQN][f / kQN] = *reinterpret_cast<const bf16x8*>(
        lds + pb[f / kQN] + h * T::kHalfB + (f % kQN) * 16 * T::kPitch);
  }
  __device__ __forceinline__ void turn(int dslot) {
    const int da = dslot * 2 * T::kHalfA, db = dslot * 2 * T::kHalfB;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      pa[kk] += da;
      pb[kk] += db;
    }
  }
  __device__ __forceinline__ void mfma(int i, int j, int r, int c, int kk) {
    acc[kQM * i + r][kQN * j + c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        bf[j][c][kk], af[i][r][kk], acc[kQM * i + r][kQN * j + c], 0, 0, 0);
  }
  template <int N>
  __device__ __forceinline__ void wait_vm() {
    fqa::wait_vm<N>();
  }
  template <int N>
  __device__ __forceinline__ void wait_lgkm() {
    static_assert(N >= 0 && N < 16, "lgkmcnt");
    __builtin_amdgcn_s_waitcnt(0xC07F | N << 8);
  }
  __device__ __forceinline__ void barrier() { fqa::barrier(); }
  __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
};

template <class T, bool kNT, bool kF32Out, bool kPartial, bool kArgmax = false, bool kAppend = false>
__global__ void __launch_bounds__(T::kThreads, 1) gemm_quad_kernel(GemmArgs a) {
  constexpr int dA = T::kDmaA, dB = T::kDmaB;
  using Ops = QuadOps<T, kNT>;
  __shared__ __attribute__((aligned(1024))) char lds[kGemmLds<T, kAppend>];
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;
  int tm, tn, sp;
  tile_of(a, tm, tn, sp);
  const int row0 = tm * T::kBM, col0 = tn * T::kBN;
  const int nst = a.K / T::kBK;
  const int n = (nst - sp + a.splits - 1) / a.splits;  // >= 1: splits <= steps
  Ops o;
  o.lds = lds;
  o.n = n;
  o.kstride = (long long)a.splits * T::kBK;

  // Wave w's DMA instruction i of a half covers rows 8 (w d + i) + lane / 8 (d instructions
  // per wave); a lane fills LDS chunk lane % 8 of its row, so it reads global chunk
  // (lane % 8) ^ swz(row).
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < dA; ++i) {
      const int r = 8 * (w * dA + i) + (lane >> 3);
      const int gr = min(row0 + T::kBM / 2 * h + r, a.M - 1);
      o.off_a[h][i] = (uint32_t)((long long)gr * a.ldx * 2) + ((lane & 7) ^ T::swz(r)) * 16;
    }
#pragma unroll
    for (int i = 0; i < dB; ++i) {
      const int r = 8 * (w * dB + i) + (lane >> 3);
      o.off_b[h][i] = (uint32_t)((long long)(col0 + T::kBN / 2 * h + r) * a.ldw * 2) +
                      ((lane & 7) ^ T::swz(r)) * 16;
    }
  }
  o.dst_a = lds_base + w * (dA * 1024);
  o.dst_b = lds_base + Ops::kB + w * (dB * 1024);
  // one row tile, unsplit, up to 128 rows: W streams from HBM
  constexpr bool kSeg = kNT && T::kBM == 128;
  const Segments segs{n, kSeg ? (int)(blockIdx.x >> 3) & 3 : 0};
  o.pos = segs.first();
  o.xs = a.x + (long long)sp * T::kBK + o.pos * o.kstride;
  o.ws = a.w + (long long)sp * T::kBK + o.pos * o.kstride;
  QuadSchedule<T> schedule;
  schedule.stage_first(o, n);

  // fragment (r, kk) of a half: row (wave's first) + 16 r + lane % 16, 16-byte chunk
  // 4 kk + lane / 16
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int c = ((4 * kk + (lane >> 4)) ^ T::swz(lane & 15)) * 16;
    o.pa[kk] = (wm * (T::kBM / 4) + (lane & 15)) * T::kPitch + c;
    o.pb[kk] = Ops::kB + (wn * (T::kBN / 4) + (lane & 15)) * T::kPitch + c;
  }
  auto& acc = o.acc;
#pragma unroll
  for (int rb = 0; rb < T::kTM; ++rb)
#pragma unroll
    for (int cb = 0; cb < T::kTN; ++cb) acc[rb][cb] = float4_t{0.f, 0.f, 0.f, 0.f};
  schedule.read_first(o);
  auto steps = [&](int end) { schedule.steps(o, n, end); };
  if constexpr (kSeg)
    run_segments(segs, acc, steps);
  else
    steps(n);
  wait_vm<0>();  // the DMAs past the end: the LDS is reused or given back

  // the epilogue's addresses are computed after the loop, not held in registers through it
  int elane = lane, erow0 = row0, ecol0 = col0;
  asm volatile("" : "+v"(elane), "+s"(erow0), "+s"(ecol0));
  // ... and the accumulators stay in AGPRs up to here (VALU ops cannot read those: without
  // this the allocator spreads the epilogue's copies into the loop and spills)
  if constexpr (T::kTM * T::kTN >= 64) {
#pragma unroll
    for (int rb = 0; rb < T::kTM; ++rb)
#pragma unroll
      for (int cb = 0; cb < T::kTN; ++cb) asm volatile("" : "+a"(acc[rb][cb]));
  }
  tile_epilogue<T, kF32Out, kPartial, kArgmax, kAppend>(a, lds, acc, erow0, ecol0, tn, sp, wm, wn, w,
                                                        elane);
}

// A few rows: no K split over workgroups and no reduction launch.  A workgroup takes a tile of
// kBM x kBN outputs over the whole of K, each of its waves a contiguous part of the k steps,
// staged through a ring of kSlots steps in LDS of the wave's own, so the loop has no barrier;
// the waves' fp32 sums meet in LDS at the end, added in wave order.  Tiles are small enough
// that one round of workgroups covers the CUs (o_proj at 6 rows: 8 x 16).
//  * A step's blocks of 16 rows are consumed as they land: block b is read, block b - 1's LDS
//    is refilled with its rows of step t + kSlots and (x blocks) its MFMAs issue, so nearly
//    the whole ring stays in flight.
//  * What bounds it: HBM for W and the launch at a few rows (o_proj at 6 rows 9.1 us against
//    7.4 for its W stream alone), the rate at which a CU stages x from L2 above (60-70 KB/us).
//  * W cold, against the K-split tiles and their reduction: o_proj at 6 / 32 / 100 / 250 rows
//    14.1 / 14.7 / 18.5 / 23.3 -> 8.9 / 10.6 / 14.7 / 19.4 us, qkv at 6 / 32 / 100 rows 15.6 /
//    16.2 / 19.7 -> 11.2 / 12.8 / 17.6, down at 6 / 64 rows 27.3 / 32.1 -> 21.0 / 27.3.
template <int kXB8_, int kWB8_, int kWaves_>
struct Slab {
  static constexpr int kXB8 = kXB8_, kWB8 = kWB8_, kWaves = kWaves_, kThreads = 64 * kWaves_;
  static constexpr int kBM = 8 * kXB8, kBN = 8 * kWB8;  // both staged 8 rows per DMA
  static constexpr int kMB = (kXB8 + 1) / 2, kNB = (kWB8 + 1) / 2;  // 16 x 16 blocks
  static constexpr int kSlot = (kBM + kBN) * 128;      // one step: 64 k of every row
  // an odd kXB8's last block reads 8 rows past the slot (never stored): 1 KiB more
  static constexpr int kPad = kXB8 % 2 * 1024;
  static constexpr int kFit = (160 * 1024 - kPad) / kWaves / kSlot;
  static constexpr int kDma = kXB8 + kWB8;
  static constexpr int kMost = 60 / kDma < 6 ? 60 / kDma : 6;  // vmcnt counts to 63
  static constexpr int kSlots = kFit < kMost ? kFit : kMost;
  // DMA instructions (8 rows each) of block b of a step: 16 W rows (b < kNB), then 16 x rows
  __host__ __device__ static constexpr int dmas(int b) {
    return (b < kNB ? 2 * b + 2 <= kWB8 : 2 * (b - kNB) + 2 <= kXB8) ? 2 : 1;
  }
  static constexpr int kRed = kWaves * kMB * kNB * 1024;  // the waves' sums
  static constexpr int kRingBytes = kWaves * kSlots * kSlot + kPad;
  static constexpr int kLds = kRingBytes > kRed ? kRingBytes : kRed;
  static_assert(kSlots >= 2 && kLds <= 160 * 1024 && kSlots * kDma < 64, "ring");
};

// f(integral_constant<int, b>) for every block of a step, unrolled.
template <class T, int b = 0, class F>
__device__ __forceinline__ void slab_blocks(F&& f) {
  if constexpr (b < T::kNB + T::kMB) {
    f(std::integral_constant<int, b>{});
    slab_blocks<T, b + 1>(f);
  }
}

template <class T, bool kF32Out, bool kPartial>
__global__ void __launch_bounds__(T::kThreads, 1) gemm_slab_kernel(GemmArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[T::kLds];
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn, sp;
  tile_of(a, tm, tn, sp);
  const int row0 = tm * T::kBM, col0 = tn * T::kBN;
  // the wave's k steps: part w of the workgroup's part sp
  const int nst = a.K / 64, parts = T::kWaves * a.splits, part = sp * T::kWaves + w;
  const int s0 = part * nst / parts, n = (part + 1) * nst / parts - s0;
  auto swz = [](int r) { return (r >> 1) & 7; };
  // slot: W rows, then x rows, 128 bytes each, chunk c of row r at c ^ swz(r)
  uint32_t off_w[T::kWB8], off_x[T::kXB8];
#pragma unroll
  for (int i = 0; i < T::kWB8; ++i) {
    const int r = 8 * i + (lane >> 3);
    off_w[i] = (uint32_t)((long long)(col0 + r) * a.ldw * 2) + ((lane & 7) ^ swz(r)) * 16;
  }
#pragma unroll
  for (int i = 0; i < T::kXB8; ++i) {
    const int r = 8 * i + (lane >> 3);
    off_x[i] = (uint32_t)((long long)min(row0 + r, a.M - 1) * a.ldx * 2) + ((lane & 7) ^ swz(r)) * 16;
  }
  float4_t acc[T::kMB][T::kNB];
#pragma unroll
  for (int rb = 0; rb < T::kMB; ++rb)
#pragma unroll
    for (int cb = 0; cb < T::kNB; ++cb) acc[rb][cb] = float4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t ring = w * (T::kSlots * T::kSlot);
  int pw[2];  // fragment kk of block b: row 16 b + lane % 16, chunk 4 kk + lane / 16
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
    pw[kk] = ring + (lane & 15) * 128 + ((4 * kk + (lane >> 4)) ^ swz(lane & 15)) * 16;
  if (n > 0) {
    const uint16_t* xs = a.x + (long long)s0 * 64;
    const uint16_t* ws = a.w + (long long)s0 * 64;
    int left = n - 1;  // steps after the one that xs and ws point at
    constexpr int kBlocks = T::kNB + T::kMB;
    auto stage = [&](int slot, int b) {
      const uint32_t dst = lds_base + ring + slot * T::kSlot;
#pragma unroll
      for (int i = 0; i < T::dmas(b); ++i) {
        const int q = b < T::kNB ? 2 * b + i : 2 * (b - T::kNB) + i;
        if (b < T::kNB) {
          dma16(ws, off_w[q], dst + q * 1024);
        } else {
          dma16(xs, off_x[q], dst + (T::kWB8 + q) * 1024);
        }
      }
    };
    // the next step; past the end the last one is staged again (never read), so that every
    // wait count holds
    auto advance = [&]() {
      const int d = left > 0 ? 64 : 0;
      --left;
      xs += d;
      ws += d;
    };
#pragma unroll
    for (int k = 0; k < T::kSlots; ++k) {
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) stage(k, b);
      advance();
    }
    int slot = 0;
    for (int t = 0; t < n; ++t) {
      const char* sb = lds + slot * T::kSlot;
      bf16x8 wf[T::kNB][2], xf[2][2];
      // block b: its fragments in registers, so its LDS is refilled; an x block's MFMAs
      auto finish = [&](int b) {
        asm volatile("" ::: "memory");
        stage(slot, b);
        if (b >= T::kNB) {
          const int rb = b - T::kNB;
#pragma unroll
          for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int cb = 0; cb < T::kNB; ++cb)
              acc[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[cb][kk], xf[rb & 1][kk],
                                                                    acc[rb][cb], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      constexpr int kAll = T::kSlots * T::kDma;
      auto read = [&](int b, auto wait_tag) {
        // block b's DMAs have landed: newer are the rest of the ring and the blocks of step
        // t + kSlots staged so far (up to b - 2)
        wait_vm<decltype(wait_tag)::value>();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          if (b < T::kNB)
            wf[b][kk] = *reinterpret_cast<const bf16x8*>(sb + pw[kk] + b * 2048);
          else
            xf[(b - T::kNB) & 1][kk] = *reinterpret_cast<const bf16x8*>(
                sb + pw[kk] + T::kWB8 * 1024 + (b - T::kNB) * 2048);
        }
      };
      slab_blocks<T>([&](auto tag) {
        constexpr int b = decltype(tag)::value;
        constexpr int d0 = T::dmas(b), d1 = b > 0 ? T::dmas(b > 0 ? b - 1 : 0) : 0;
        read(b, std::integral_constant<int, kAll - d0 - d1>{});
        if constexpr (b > 0) {
          __builtin_amdgcn_s_waitcnt(0xC27F);  // lgkmcnt(2): block b - 1's fragments
          finish(b - 1);
        }
      });
      __builtin_amdgcn_s_waitcnt(0xC07F);
      finish(kBlocks - 1);
      advance();
      slot = slot + 1 == T::kSlots ? 0 : slot + 1;
    }
  }
  wait_vm<0>();  // every DMA has landed: the LDS is reused
  __syncthreads();
#pragma unroll
  for (int rb = 0; rb < T::kMB; ++rb)
#pragma unroll
    for (int cb = 0; cb < T::kNB; ++cb)
      *reinterpret_cast<float4_t*>(lds + ((w * T::kMB + rb) * T::kNB + cb) * 1024 + lane * 16) =
          acc[rb][cb];
  __syncthreads();
  // thread -> (row, 4 columns), consecutive threads along a row
  constexpr int kRow4 = T::kBN / 4;
  for (int e = threadIdx.x; e < T::kBM * kRow4; e += T::kThreads) {
    const int r = e / kRow4, c = e % kRow4 * 4;
    const int m = row0 + r;
    if (m >= a.M) break;
    const char* src = lds + ((r >> 4) * T::kNB + (c >> 4)) * 1024 + ((r & 15) + ((c & 15) >> 2) * 16) * 16;
    float4_t v = *reinterpret_cast<const float4_t*>(src);
#pragma unroll
    for (int k = 1; k < T::kWaves; ++k)
      v += *reinterpret_cast<const float4_t*>(src + k * T::kMB * T::kNB * 1024);
    const int nc = col0 + c;
    if (kPartial)
      *reinterpret_cast<float4_t*>(a.part + ((long long)sp * a.M + m) * a.N + nc) = v;
    else if (kF32Out)
      *reinterpret_cast<float4_t*>(static_cast<float*>(a.y) + m * a.ldy + nc) = v;
    else
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.y) + m * a.ldy + nc) =
          make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
}

// The QKV projection's epilogue fused with the per-head norm + RoPE + paged append
// (fqa_qknorm_rope_append on the tile's rows, same results bit for bit): the tile's
// values are rounded to bf16 (what fqa_gemm would write) and staged in LDS, then
//  * q / k tiles: one 16-lane group per (row, head) runs norm_rope_head on the row's
//    head (the append kernel's lane layout and arithmetic), q goes to qkv, k to its page
//    (and to qkv with write_k); rows without a RoPE table row keep the projection's values;
//  * v tiles: a page whose 16 rows are all in the tile is written by its first row as
//    whole V^T rows (a register transpose of the 16 staged rows); other rows store their
//    token's column.
// v is not written to qkv.  Rows at or past meta[FQA_META_ROWS] are not written.
// What bounds it: latency, with one wave per SIMD.  One head's norm after the other (xor
// shuffles through LDS in each) and one wave walking all of a V tile's pages cost 12-25 us a
// tile; with a batch's norms side by side, DPP sums and each wave's rows settled by a lane
// each, QKV + append with 512-token prompts at 500 / 700 / 1000 / 2048 / 8192 rows 49 / 73 /
// 76 / 107 / 333 -> 40 / 53 / 57 / 92 / 309 us.  Rows on pages of their own are bound by the
// CUs that hold V, a lane's 2-byte store per clock (dims in a row; every other dim per store
// took 1.4 times that): 260 / 500 / 700 / 2048 rows 43 / 52 / 72 / 137 -> 39 / 49 / 63 / 127.
template <class T>
__device__ void append_epilogue(const GemmArgs& a, char* lds, const typename T::Block (&acc)[T::kTM][T::kTN],
                                int row0, int col0, int wm, int wn, int w, int lane) {
  constexpr int kTP = kTilePitch<T>;
  constexpr int kNH = T::kBN / kD;  // heads in the tile
  const GemmAppend& p = a.app;
  int* s_pos = reinterpret_cast<int*>(lds + T::kBM * kTP);
  int* s_slot = s_pos + T::kBM;
  const int T_rows = min(p.meta[FQA_META_ROWS], a.M);
  // the rows' positions and slots, loaded while the tile goes to LDS (position -1: no such
  // row; slot -1: nothing to append)
  int my_pos = -1, my_slot = -1;
  if (threadIdx.x < T::kBM && row0 + (int)threadIdx.x < T_rows) {
    my_pos = p.positions[row0 + threadIdx.x];
    my_slot = p.slots[row0 + threadIdx.x];
    if (my_pos < 0 || my_pos >= p.rope_max_pos || my_slot < 0 || my_slot / kPage >= p.pool_pages)
      my_slot = -1;
  }
  stage_tile<T>(lds, acc, wm, wn, lane);
  if (threadIdx.x < T::kBM) {
    s_pos[threadIdx.x] = my_pos;
    s_slot[threadIdx.x] = my_slot;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  barrier();

  const int head0 = col0 / kD;
  uint16_t* qkv = static_cast<uint16_t*>(a.y);
  if (head0 < kHq + kHkv) {  // q or k heads (a tile never mixes kinds: 4096, 5120 | kBN)
    const int g = lane >> 4, j = lane & 15;
    const bool is_k = head0 >= kHq;
    const float* wv = is_k ? p.wk : p.wq;
    const float4 w1 = *reinterpret_cast<const float4*>(wv + 4 * j);
    const float4 w2 = *reinterpret_cast<const float4*>(wv + 64 + 4 * j);
    const float wa[4] = {w1.x, w1.y, w1.z, w1.w}, wb[4] = {w2.x, w2.y, w2.z, w2.w};
    // (row, head) pairs in batches of kB per lane group: every load of a batch (staged
    // values, positions, then the cos/sin rows) is issued before any is used, and the batch's
    // norms run side by side, before any of its stores: a SIMD has one wave here, so one
    // head's chain after the other is all latency
    constexpr int kPerGroup = T::kBM * kNH / (T::kWaves * 4);
    constexpr int kB = kPerGroup / ((kPerGroup + 15) / 16);
    static_assert(kPerGroup % kB == 0, "batches");
    for (int b0 = 0; b0 < kPerGroup; b0 += kB) {
      int rt[kB], pos[kB];
      uint2 lo[kB], hv[kB], olo[kB], ohi[kB];
      float4 c4[kB], s4[kB];
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int hr = (b0 + b) * T::kWaves * 4 + w * 4 + g;  // (row, head) of this group
        rt[b] = hr / kNH;
        const int hi = hr % kNH;
        pos[b] = s_pos[rt[b]];
        const char* src = lds + rt[b] * kTP + (hi * kD + 4 * j) * 2;
        lo[b] = *reinterpret_cast<const uint2*>(src);
        hv[b] = *reinterpret_cast<const uint2*>(src + 128);
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int pc = pos[b] >= 0 && pos[b] < p.rope_max_pos ? pos[b] : 0;
        c4[b] = *reinterpret_cast<const float4*>(p.cos_tab + (long long)pc * 64 + 4 * j);
        s4[b] = *reinterpret_cast<const float4*>(p.sin_tab + (long long)pc * 64 + 4 * j);
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const float cs[4] = {c4[b].x, c4[b].y, c4[b].z, c4[b].w};
        const float sn[4] = {s4[b].x, s4[b].y, s4[b].z, s4[b].w};
        norm_rope_head(lo[b], hv[b], wa, wb, cs, sn, p.eps, olo[b], ohi[b]);  // all lanes
      }
#pragma unroll
      for (int b = 0; b < kB; ++b) {
        const int hr = (b0 + b) * T::kWaves * 4 + w * 4 + g;
        const int row = row0 + rt[b], head = head0 + hr % kNH;
        const bool pos_ok = pos[b] >= 0 && pos[b] < p.rope_max_pos;  // false: no such row too
        if (row >= T_rows) continue;
        if (!pos_ok) {  // no table row: the projection's values, as unfused
          olo[b] = lo[b];
          ohi[b] = hv[b];
        }
        if (!is_k || p.write_k) {
          uint16_t* d = qkv + (long long)row * a.ldy + head * kD + 4 * j;
          *reinterpret_cast<uint2*>(d) = olo[b];
          *reinterpret_cast<uint2*>(d + 64) = ohi[b];
        }
        const int slot = s_slot[rt[b]];
        if (is_k && slot >= 0) {
          uint16_t* kd = p.pool + run_offset(slot / kPage, head - kHq) + (slot % kPage) * kD + 4 * j;
          *reinterpret_cast<uint2*>(kd) = olo[b];
          *reinterpret_cast<uint2*>(kd + 64) = ohi[b];
        }
      }
    }
    return;
  }
  // v heads.  Each wave takes kBM / 4 rows in a row; lane l first settles row l: skipped,
  // written as a whole page, or its column.
  constexpr int kRows = T::kBM / T::kWaves;
  static_assert(kRows <= kWave && kRows % kPage == 0, "a lane per row");
  const int rt = w * kRows + min(lane, kRows - 1);
  const int slot = s_slot[rt];
  const int tok = slot % kPage, lt = rt - tok;  // the page's first row, in the tile
  const bool valid = lane < kRows && slot >= 0;
  // A page whose 16 rows all lie in the tile, each in its place, is written by its first row;
  // any other row writes its own column.
  const bool inside = valid && lt >= 0 && lt + kPage <= T::kBM;
  const int* first = s_slot + (inside ? lt : 0);
  int off = 0;  // (every read is on its way before the first is looked at)
#pragma unroll
  for (int i = 0; i < kPage; ++i) off |= first[i] ^ (slot - tok + i);
  const bool whole = inside && off == 0;
  const int kvh0 = head0 - kHq - kHkv;
  // whole pages: lane l holds dims 2l, 2l+1 of each head
  for (uint64_t m = __ballot(whole && tok == 0); m; m &= m - 1) {
    const int l = __ffsll((unsigned long long)m) - 1, r = w * kRows + l;
    const long long page = __builtin_amdgcn_readlane(slot, l) / kPage;
#pragma unroll
    for (int hi = 0; hi < kNH; ++hi) {
      uint16_t* vt = p.pool + run_offset(page, kvh0 + hi) + kVOff + 2 * lane * kPage;
      uint32_t x[kPage];
#pragma unroll
      for (int t = 0; t < kPage; ++t)
        x[t] = *reinterpret_cast<const uint32_t*>(lds + (r + t) * kTP + (hi * kD + 2 * lane) * 2);
      uint32_t y0[8], y1[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        y0[k] = __builtin_amdgcn_perm(x[2 * k + 1], x[2 * k], 0x05040100u);
        y1[k] = __builtin_amdgcn_perm(x[2 * k + 1], x[2 * k], 0x07060302u);
      }
      uint4* v4 = reinterpret_cast<uint4*>(vt);
      v4[0] = make_uint4(y0[0], y0[1], y0[2], y0[3]);
      v4[1] = make_uint4(y0[4], y0[5], y0[6], y0[7]);
      v4[2] = make_uint4(y1[0], y1[1], y1[2], y1[3]);
      v4[3] = make_uint4(y1[4], y1[5], y1[6], y1[7]);
    }
  }
  for (uint64_t m = __ballot(valid && !whole); m; m &= m - 1) {
    const int l = __ffsll((unsigned long long)m) - 1, r = w * kRows + l;
    const int sl = __builtin_amdgcn_readlane(slot, l);
    // here lane l holds dims l and 64 + l: a store's 64 places lie in 2 KiB in a row
#pragma unroll
    for (int hi = 0; hi < kNH; ++hi) {
      const uint16_t* x = reinterpret_cast<const uint16_t*>(lds + r * kTP) + hi * kD + lane;
      uint16_t* vt = p.pool + run_offset(sl / kPage, kvh0 + hi) + kVOff + lane * kPage + sl % kPage;
      vt[0] = x[0];
      vt[kWave * kPage] = x[kWave];
    }
  }
}

// Row m's token: the largest of its per-tile maxima, ties in the reference's greedy order
// (greedy_key).  One wave per row.
__global__ void __launch_bounds__(256) gemm_argmax_reduce_kernel(GemmArgs a, int32_t* out) {
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (m >= a.M) return;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  const float* rv = a.amax_v + (long long)m * a.n_tiles;
  const int* ri = a.amax_i + (long long)m * a.n_tiles;
  // 8 tiles per lane per round, all loads issued before any compare (clamped indices;
  // the repeats of the last tile change nothing)
  for (int t0 = 0; t0 < a.n_tiles; t0 += 8 * kWave) {
    float v[8];
    int i[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t = min(t0 + k * kWave + lane, a.n_tiles - 1);
      v[k] = rv[t];
      i[k] = ri[t];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (v[k] > bv || (v[k] == bv && greedy_key(i[k]) < greedy_key(bi))) {
        bv = v[k];
        bi = i[k];
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, kWave);
    const int oi = __shfl_xor(bi, o, kWave);
    if (ov > bv || (ov == bv && greedy_key(oi) < greedy_key(bi))) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane == 0) out[m] = bv > kGreedyFloor ? bi : 0;  // nothing above -1e30: 0, as fqa_sample
}

// y = sum over the splits of the fp32 partials, 4 columns per thread.
template <bool kF32Out>
__global__ void __launch_bounds__(256) gemm_reduce_kernel(GemmArgs a) {
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;  // float4 index
  const int n4 = a.N / 4;
  if (q >= (long long)a.M * n4) return;
  const int m = (int)(q / n4), n = (int)(q % n4) * 4;
  const long long plane = (long long)a.M * a.N;
  float4 s = *reinterpret_cast<const float4*>(a.part + (long long)m * a.N + n);
  for (int k = 1; k < a.splits; ++k) {
    const float4 v = *reinterpret_cast<const float4*>(a.part + k * plane + (long long)m * a.N + n);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  if (kF32Out) {
    *reinterpret_cast<float4*>(static_cast<float*>(a.y) + m * a.ldy + n) = s;
  } else {
    const uint2 p = make_uint2(pack_bf16x2(s.x, s.y), pack_bf16x2(s.z, s.w));
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.y) + m * a.ldy + n) = p;
  }
}

bool gemm_shape_ok(int M, int N, int K) {
  return M >= 0 && N > 0 && K > 0 && N % 128 == 0 && K % kGK == 0;
}

// K splits that fqa_gemm_workspace_bytes has room for at least (a fixed rule, so that a
// workspace sized once stays valid): as many as bring tiles of 32, 64, 128 or 256 rows (the
// fewest that cover M, 256 above) by 128 columns (256 above 1024 rows) to the 256 CUs once,
// at most 16, one where 160 tiles or more exist.
int sized_splits(int M, int N, int K) {
  int bm = M > 128 ? 256 : M > 64 ? 128 : M > 32 ? 64 : 32;
  const int bn = M > 1024 && N % 256 == 0 ? 256 : 128;
  if (M > 128 && M <= 256 && N / 128 < 40) bm = 128;
  const int tiles = ((M + bm - 1) / bm) * (N / bn);
  int s = tiles >= 160 ? 1 : 256 / tiles;
  if (s > 16) s = 16;
  if (s > K / kGK) s = K / kGK;
  return s < 1 ? 1 : s;
}

// The slab tiles: {rows, columns} and, in slab_dispatch, their waves.
constexpr int kSlabs[][2] = {{8, 16},  {8, 24},  {16, 16}, {16, 24}, {32, 16}, {32, 24}, {32, 32},
                             {64, 32}, {64, 48}, {96, 32}, {96, 48}, {64, 64}, {96, 64}, {64, 96}};
template <class F>
bool slab_dispatch(int i, F&& f) {
  switch (i) {
    case 0: return f(Slab<1, 2, 8>{});
    case 1: return f(Slab<1, 3, 8>{});
    case 2: return f(Slab<2, 2, 8>{});
    case 3: return f(Slab<2, 3, 8>{});
    case 4: return f(Slab<4, 2, 4>{});
    case 5: return f(Slab<4, 3, 4>{});
    case 6: return f(Slab<4, 4, 4>{});
    case 7: return f(Slab<8, 4, 4>{});
    case 8: return f(Slab<8, 6, 4>{});
    case 9: return f(Slab<12, 4, 4>{});
    case 10: return f(Slab<12, 6, 4>{});
    case 11: return f(Slab<8, 8, 4>{});
    case 12: return f(Slab<12, 8, 4>{});
    default: return f(Slab<8, 12, 4>{});
  }
}

// The launch plan of one call.
enum Tiles { kTileT, kTileS, kTileM, kTileH, kTileQ, kTileP, kTileL, kSlab0 };
struct GemmPlan {
  int tile;  // Tiles; kSlab0 + i: kSlabs[i]
  int bm, bn, splits, m_tiles, n_tiles;
};

// Chosen by a model of the time in us, fitted to measurements with W cold on 6144 x 4096, 4096 x
// 4096, 24576 x 4096 and 4096 x 12288 at 6 to 2048 rows (within ~15% of each, and nearly always
// the measured order), and checked on 22 widths from 128 to 24576 by 128 to 12288 k at 1 to
// 1024 rows (4554 shapes: the plan is 2.5% behind the best of all plans on average):
//  * Tiles of 128 columns or more: 2.4 for the launch and, per round of 256 workgroups, 5 to
//    start and store and, per step of 64 k, 1.29 (256 x 256), 1.03 (192 x 256, 256 x 192; 1.24
//    with K split), 0.78 (256 x 128) or 0.45 (128 x 128; 0.58 with K split, 0.75 with a single
//    row tile unsplit, whose W comes from HBM).  What decides between them is mostly how full
//    the last round is: gate_up at 384 / 700 / 1000 / 1500 rows 90 / 154 / 178 / 260 us without
//    the 192-wide tiles, 80 / 141 / 164 / 238 with them; qkv at 1500 rows 77 -> 68, down 139 ->
//    127.
//  * A K split by a multiple of four at up to 256 rows: 15% more per step, its workgroups
//    meeting on the same HBM channels (down at 160 / 200 / 256 rows, 256 x 128, 8 parts 41.8 /
//    42.7 / 47.2 us, 7 parts 35.4 / 37.2 / 39.7).
//  * Slabs: 6, 1 per 64 KB that a workgroup stages and 1 per 4096 outputs of the tile (the
//    sum over its waves); one round of workgroups; for x that fits an XCD's L2
//    beside the W stream (3.5 MB: at 12288 k and 160 rows the slabs lose).
//  * A K split adds the reduction: 2.5 (3 to a slab), 1 per split and 1 per million fp32
//    partials (8 MB).
// Up to 128 rows with more than 128 column tiles (gate_up, lm_head), where K cannot be split
// over the CUs left, the smallest tile that covers M streams W once at HBM's rate (18944 x 1024
// at 4 / 64 rows 11.5 / 13.5 us, in 128 x 128 tiles 14.0 / 15.8).
// max_splits bounds K splits; 1 (fqa_gemm_argmax, and shapes whose workspace is empty) also
// leaves the slabs out, so that equal shapes sum in the same order.
GemmPlan gemm_plan(int M, int N, int K, int max_splits) {
  const int nst = K / kGK;
  auto make = [&](int tile, int bm, int bn, int s) {
    return GemmPlan{tile, bm, bn, s, (M + bm - 1) / bm, N / bn};
  };
  if (M <= 128 && N / 128 > 128)
    return M > 64 ? make(kTileM, 128, 128, 1) : M > 32 ? make(kTileS, 64, 128, 1) : make(kTileT, 32, 128, 1);
  // The QKV width at 489..512 rows of 4096 k or more, where the call may split: K in two, and
  // the append kernel reads the two planes.  With the append in the epilogue of 128 x 128 tiles,
  // decode rows on their own pages keep the few CUs that hold V busy after all others; prompts
  // and fqa_gemm, which has to share the plan so that fused and unfused agree, are faster
  // unsplit.  Split / unsplit, 4096 k (us):
  //   rows               464          484          488          496          512
  //   own pages      44.9 / 46.9  45.4 / 48.6  45.1 / 48.9  45.5 / 49.8  45.4 / 50.5
  //   512-token prompts  43.9 / 38.3  44.1 / 39.5  44.0 / 40.0  44.2 / 40.4  44.2 / 41.2
  //   fqa_gemm       40.5 / 36.2  41.0 / 37.9  40.8 / 37.8  40.8 / 38.3  40.6 / 38.8
  // With fewer k the split costs more (512 rows of 3072 k: 39.0 / 41.2, 37.4 / 31.1, 33.7 / 29.0;
  // of 1024 k: 27.9 / 25.4, 26.1 / 14.5, 22.5 / 12.5).
  if (N == kQkvStride && M > 488 && M <= 512 && K >= 4096 && max_splits > 1)
    return make(kTileH, 256, 128, 2);
  GemmPlan best{};
  float best_us = 3.4e38f;
  auto consider = [&](const GemmPlan& p, float us) {
    if (p.splits > 1) us += 2.5f + p.splits + 1e-6f * p.splits * M * N;
    if (us < best_us) {
      best_us = us;
      best = p;
    }
  };
  // (256 x 192 tiles cut heads: not at the QKV width, whose epilogue may append)
  const struct {
    int tile, bm, bn;
    float step, split_step;
  } quads[] = {{kTileL, 256, 256, 1.29f, 1.29f},
               {kTileP, 192, 256, 1.03f, 1.24f},
               {kTileQ, 256, 192, 1.03f, 1.24f},
               {kTileH, 256, 128, 0.78f, 0.78f},
               {kTileM, 128, 128, 0.45f, 0.58f}};
  for (const auto& q : quads) {
    if (N % q.bn || (q.tile == kTileQ && N == kQkvStride)) continue;
    for (int s = 1; s <= max_splits && s <= 16 && s <= nst; ++s) {
      const GemmPlan p = make(q.tile, q.bm, q.bn, s);
      const long long g = (long long)p.m_tiles * p.n_tiles * s;
      if (s > 1 && g > 256) break;
      float step = s > 1 ? q.split_step : q.tile == kTileM && p.m_tiles == 1 ? 0.75f : q.step;
      if (s > 1 && s % 4 == 0 && M <= 256) step *= 1.15f;
      consider(p, 2.4f + (float)((g + 255) / 256) * ((float)((nst + s - 1) / s) * step + 5.f));
    }
  }
  if (max_splits > 1 && (long long)M * K * 2 <= 3500000) {
    for (int i = 0; i < (int)(sizeof(kSlabs) / sizeof(kSlabs[0])); ++i) {
      const int bm = kSlabs[i][0], bn = kSlabs[i][1];
      if (N % bn) continue;
      for (int s = 1; s <= 4 && s <= max_splits && s <= nst; s *= 2) {
        const GemmPlan p = make(kSlab0 + i, bm, bn, s);
        if ((long long)p.m_tiles * p.n_tiles * s > 256) break;
        consider(p, (s > 1 ? 6.5f : 6.f) + (bm + bn) * 2.f * K / s / 64e3f + bm * bn / 4096.f);
      }
    }
  }
  return best;
}

// The largest K split a call may use: what the shape's workspace is sized for, and beyond
// that (not for the QKV width, whose size is fixed by sized_splits) what the plan would take
// if `bytes` has room.
int splits_allowed(int M, int N, int K, int64_t bytes) {
  const int s = sized_splits(M, N, K);
  if (s == 1 || N == kQkvStride) return s;
  const int64_t fit = bytes / ((int64_t)M * N * 4);
  return fit > 16 ? 16 : fit > s ? (int)fit : s;
}

// f(kNT) for an unsplit launch of a quad tile: one row tile of 128 columns streams W from HBM
// (and on 128 x 128 takes K in segments).  Every form of a call goes by this rule, so that
// fqa_gemm, fqa_gemm_argmax and the append's epilogue sum a shape in one order.
template <class T, class F>
void unsplit_quad(const GemmArgs& a, F&& f) {
  if constexpr (T::kBN == 128) {
    if (a.m_tiles == 1) return f(std::true_type{});
  }
  f(std::false_type{});
}
template <class T>
void launch_gemm(const GemmArgs& a, bool f32, hipStream_t st) {
  const dim3 grid((unsigned)(a.m_tiles * a.n_tiles * a.splits));
  const dim3 block(T::kThreads);
  if constexpr (kIsQuad<T>) {
    if (a.splits > 1)
      hipLaunchKernelGGL((gemm_quad_kernel<T, false, false, true>), grid, block, 0, st, a);
    else
      unsplit_quad<T>(a, [&](auto nt) {
        if (f32)
          hipLaunchKernelGGL((gemm_quad_kernel<T, decltype(nt)::value, true, false>), grid, block, 0, st, a);
        else
          hipLaunchKernelGGL((gemm_quad_kernel<T, decltype(nt)::value, false, false>), grid, block, 0, st, a);
      });
  } else if (f32) {
    hipLaunchKernelGGL((gemm_kernel<T, true>), grid, block, 0, st, a);
  } else {
    hipLaunchKernelGGL((gemm_kernel<T, false>), grid, block, 0, st, a);
  }
}
template <class T>
void launch_argmax(const GemmArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(a.m_tiles * a.n_tiles));
  const dim3 block(T::kThreads);
  if constexpr (!kIsQuad<T>)
    hipLaunchKernelGGL((gemm_kernel<T, false, true>), grid, block, 0, st, a);
  else
    unsplit_quad<T>(a, [&](auto nt) {
      hipLaunchKernelGGL((gemm_quad_kernel<T, decltype(nt)::value, false, false, true>), grid, block, 0, st, a);
    });
}
template <class T>
void launch_append(const GemmArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(a.m_tiles * a.n_tiles));
  const dim3 block(T::kThreads);
  unsplit_quad<T>(a, [&](auto nt) {
    hipLaunchKernelGGL((gemm_quad_kernel<T, decltype(nt)::value, false, false, false, true>), grid, block, 0, st, a);
  });
}
// A slab's launch; planes: fp32 into a.part also without a split.
template <class T>
void launch_slab(const GemmArgs& a, bool f32, bool planes, hipStream_t st) {
  const dim3 grid((unsigned)(a.m_tiles * a.n_tiles * a.splits));
  const dim3 block(T::kThreads);
  if (planes)
    hipLaunchKernelGGL((gemm_slab_kernel<T, false, true>), grid, block, 0, st, a);
  else if (f32)
    hipLaunchKernelGGL((gemm_slab_kernel<T, true, false>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((gemm_slab_kernel<T, false, false>), grid, block, 0, st, a);
}
}  // namespace
}  // namespace fqa

using namespace fqa;

extern "C" int64_t fqa_gemm_workspace_bytes(int32_t M, int32_t N, int32_t K) {
  if (!gemm_shape_ok(M, N, K) || M == 0) return 0;
  const int sized = sized_splits(M, N, K);
  if (sized == 1) return 0;
  const int most = splits_allowed(M, N, K, INT64_MAX);
  const int want = gemm_plan(M, N, K, most).splits;
  return (int64_t)(want > sized ? want : sized) * M * N * 4;
}

namespace fqa {

// Validates a call and fills the kernel arguments and plan; FQA_OK or an FQA_E code.
static int gemm_prepare(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y,
                        int64_t ldy, int32_t M, int32_t N, int32_t K, void* workspace,
                        int64_t workspace_bytes, GemmArgs& a, GemmPlan& p) {
  if (M < 0 || N <= 0 || K <= 0) return FQA_EINVAL;
  if (!gemm_shape_ok(M, N, K)) return FQA_EUNSUPPORTED;
  if (M == 0) return FQA_OK;
  if (!x || !w || !y) return FQA_EINVAL;
  if (ldx < K || ldw < K || ldy < N || ldx % 8 || ldw % 8 || ldy % 4) return FQA_EINVAL;
  if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)y & 15)) return FQA_EINVAL;
  // DMA lane offsets are 32-bit: every row start of x and W must lie within 4 GiB
  if ((int64_t)(M - 1) * ldx * 2 >= (int64_t)1 << 32 || (int64_t)(N - 1) * ldw * 2 >= (int64_t)1 << 32)
    return FQA_EUNSUPPORTED;
  const int sized = sized_splits(M, N, K);
  if (sized > 1 && (!workspace || workspace_bytes < (int64_t)sized * M * N * 4 ||
                    ((uintptr_t)workspace & 15)))
    return FQA_EINVAL;
  p = gemm_plan(M, N, K, splits_allowed(M, N, K, workspace_bytes));
  if ((int64_t)p.m_tiles * p.n_tiles * p.splits > 0x7fffffff) return FQA_EINVAL;
  a = GemmArgs{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), y, nullptr,
               ldx, ldw, ldy, M, N, K, p.splits, p.m_tiles, p.n_tiles};
  if (sized > 1) a.part = static_cast<float*>(workspace);
  return FQA_OK;
}

// planes: a slab leaves fp32 in a.part also without a split
static void gemm_launch_main(const GemmArgs& a, const GemmPlan& p, bool f32, bool planes,
                             hipStream_t st) {
  switch (p.tile) {
    case kTileL: launch_gemm<TileL>(a, f32, st); break;
    case kTileP: launch_gemm<TileP>(a, f32, st); break;
    case kTileQ: launch_gemm<TileQ>(a, f32, st); break;
    case kTileH: launch_gemm<TileH>(a, f32, st); break;
    case kTileM: launch_gemm<TileM>(a, f32, st); break;
    case kTileS: launch_gemm<TileS>(a, f32, st); break;
    case kTileT: launch_gemm<TileT>(a, f32, st); break;
    default:
      slab_dispatch(p.tile - kSlab0, [&](auto t) {
        launch_slab<decltype(t)>(a, f32, planes || a.splits > 1, st);
        return true;
      });
  }
}

int gemm_launch_partials(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y,
                         int64_t ldy, int32_t M, int32_t N, int32_t K, void* workspace,
                         int64_t workspace_bytes, hipStream_t st, const GemmAppend& app,
                         bool* appended) {
  GemmArgs a;
  GemmPlan p;
  *appended = false;
  const int rc = gemm_prepare(x, ldx, w, ldw, y, ldy, M, N, K, workspace, workspace_bytes, a, p);
  if (rc != FQA_OK || M == 0) return rc;
  if (p.splits == 1 && p.tile < kSlab0) {  // (48 column tiles: never a 32- or 64-row tile)
    a.app = app;
    if (p.tile == kTileL)
      launch_append<TileL>(a, st);
    else if (p.tile == kTileP)
      launch_append<TileP>(a, st);
    else if (p.tile == kTileH)
      launch_append<TileH>(a, st);
    else
      launch_append<TileM>(a, st);
    *appended = true;
    return 0;
  }
  gemm_launch_main(a, p, false, true, st);
  return p.splits;
}

}  // namespace fqa

extern "C" int fqa_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y,
                        int64_t ldy, int32_t M, int32_t N, int32_t K, int32_t y_f32,
                        void* workspace, int64_t workspace_bytes, void* stream) {
  GemmArgs a;
  GemmPlan p;
  const int rc = gemm_prepare(x, ldx, w, ldw, y, ldy, M, N, K, workspace, workspace_bytes, a, p);
  if (rc != FQA_OK || M == 0) return rc;
  hipStream_t st = (hipStream_t)stream;
  gemm_launch_main(a, p, y_f32 != 0, false, st);
  if (p.splits > 1) {
    const long long n4 = (long long)M * (N / 4);
    const unsigned blocks = (unsigned)((n4 + 255) / 256);
    if (y_f32)
      hipLaunchKernelGGL((gemm_reduce_kernel<true>), dim3(blocks), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((gemm_reduce_kernel<false>), dim3(blocks), dim3(256), 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? FQA_OK : FQA_ELAUNCH;
}

extern "C" int64_t fqa_gemm_argmax_workspace_bytes(int32_t M, int32_t N, int32_t K) {
  // a pair per row and column tile, sized for tiles of 128 columns, above 1024 rows of 256
  if (!gemm_shape_ok(M, N, K) || M == 0) return 0;
  return (int64_t)(N / (M > 1024 && N % 256 == 0 ? 256 : 128)) * M * 8;
}

extern "C" int fqa_gemm_argmax(const void* x, int64_t ldx, const void* w, int64_t ldw,
                               int32_t M, int32_t N, int32_t K, int32_t* out, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  if (M < 0 || N <= 0 || K <= 0) return FQA_EINVAL;
  if (!gemm_shape_ok(M, N, K)) return FQA_EUNSUPPORTED;
  if (M == 0) return FQA_OK;
  if (!x || !w || !out || !workspace) return FQA_EINVAL;
  if (ldx < K || ldw < K || ldx % 8 || ldw % 8) return FQA_EINVAL;
  if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)workspace & 15)) return FQA_EINVAL;
  if ((int64_t)(M - 1) * ldx * 2 >= (int64_t)1 << 32 || (int64_t)(N - 1) * ldw * 2 >= (int64_t)1 << 32)
    return FQA_EUNSUPPORTED;
  // without a K split (every tile sees whole rows of its columns)
  GemmPlan p = gemm_plan(M, N, K, 1);
  if (M > 1024 && N % 256 == 0 && p.bn != 256)  // as the workspace is sized
    p = GemmPlan{kTileL, 256, 256, 1, (M + 255) / 256, N / 256};
  if (workspace_bytes < fqa_gemm_argmax_workspace_bytes(M, N, K)) return FQA_EINVAL;
  if ((int64_t)p.m_tiles * p.n_tiles > 0x7fffffff) return FQA_EINVAL;
  GemmArgs a{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), nullptr, nullptr,
             ldx, ldw, 0, M, N, K, 1, p.m_tiles, p.n_tiles,
             static_cast<float*>(workspace),
             reinterpret_cast<int*>(static_cast<char*>(workspace) + (int64_t)p.n_tiles * M * 4)};
  hipStream_t st = (hipStream_t)stream;
  switch (p.tile) {
    case kTileL: launch_argmax<TileL>(a, st); break;
    case kTileP: launch_argmax<TileP>(a, st); break;
    case kTileQ: launch_argmax<TileQ>(a, st); break;
    case kTileH: launch_argmax<TileH>(a, st); break;
    case kTileM: launch_argmax<TileM>(a, st); break;
    case kTileS: launch_argmax<TileS>(a, st); break;
    default: launch_argmax<TileT>(a, st); break;
  }
  hipLaunchKernelGGL(gemm_argmax_reduce_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, st, a,
                     out);
  return hipGetLastError() == hipSuccess ? FQA_OK : FQA_ELAUNCH;
}
