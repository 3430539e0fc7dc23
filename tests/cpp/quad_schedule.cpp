// quad_schedule.cpp — runs QuadSchedule (flashqwen_amd/csrc/fqa_quad_schedule.h) on the host
// with operations that record what one wave of gemm_quad_kernel does, and checks that the
// order holds whatever the waves' speeds.  All waves run the same program and meet only at its
// barriers, so an event of one wave before barrier e comes before every event of another after
// it, and nothing else is ordered between them:
//  * a half is read only behind a barrier that follows every wave's wait for its DMA;
//  * a half is refilled only behind a barrier that follows the end of every wave's reads of it
//    (a read ends where the wave waits for it: lgkmcnt, or the first MFMA that uses it);
//  * the MFMAs of step t take fragments of step t, each pair of blocks once.
// Prints the number of operations checked; exits with 1 at the first violation.
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <set>
#include <tuple>
#include <vector>

#include "../../flashqwen_amd/csrc/fqa_quad_schedule.h"

using namespace fqa;

namespace {
long g_ops = 0;

template <class T>
struct Recorder {
  struct Half {
    int step = -1;         // the k step its slot holds
    int issued = 0;        // DMA instructions of it, and those waited for
    int landed = 0;
    int landed_epoch = -1;  // barriers passed when the last one was waited for
    std::vector<int> reads;  // per read: barriers passed when it ended, -1: it has not
  };
  struct Read {
    Half* half;
    size_t index;
    int step;
  };
  const char* name;
  int n;
  int epoch = 0, at = 0, before = 0, slot = 0;
  Half halves[2][2][T::kRing];  // operand, half, slot
  std::deque<Half*> dma;
  std::deque<Read> lds;  // reads in flight (LDS reads end in order)
  Read frag[2][2][16];
  long mfmas = 0;
  std::set<std::tuple<int, int, int, int, int>> seen;

  [[noreturn]] void fail(const char* what, int op, int h) {
    std::printf("%s, %d steps: %s (%c%d, step %ld)\n", name, n, what, op ? 'B' : 'A', h, mfmas / kPerStep);
    std::exit(1);
  }
  static constexpr long kPerStep = 4 * 2 * T::kQM * T::kQN;

  void stage(int op, int h, int to, int step, int instr, int count) {
    ++g_ops;
    Half& x = halves[op][h][to];
    if (instr == 0) {
      if (x.issued != x.landed) fail("refilled while its DMA is in flight", op, h);
      for (int e : x.reads)
        if (e < 0 || e >= epoch) fail("refilled before every wave has read it", op, h);
      x = Half{};
      x.step = step;
    }
    if (x.step != step || x.issued != instr || instr >= count) fail("DMA out of order", op, h);
    ++x.issued;
    dma.push_back(&x);
  }
  void read(int op, int h, int f, int count) {
    ++g_ops;
    Half& x = halves[op][h][slot];
    if (x.issued != count || x.landed != count || x.landed_epoch >= epoch)
      fail("read before every wave's DMA has landed", op, h);
    frag[op][h][f] = Read{&x, x.reads.size(), x.step};
    x.reads.push_back(-1);
    lds.push_back(frag[op][h][f]);
  }
  void end_reads(size_t left) {
    while (lds.size() > left) {
      lds.front().half->reads[lds.front().index] = epoch;
      lds.pop_front();
    }
  }
  void use(const Read& r) {
    size_t left = lds.size();
    for (size_t i = 0; i < lds.size(); ++i)
      if (lds[i].half == r.half && lds[i].index == r.index) left = lds.size() - i - 1;
    end_reads(left);
  }

  // QuadSchedule's operations
  void stage_a(int h, int to, int i) { stage(0, h, to, at, i, T::kDmaA); }
  void stage_a1_prev(int to, int i) { stage(0, 1, to, before, i, T::kDmaA); }
  void stage_b(int h, int to, int i) { stage(1, h, to, at, i, T::kDmaB); }
  void keep() { before = at; }
  void advance(bool more) { at += more; }
  void read_a(int h, int f) { read(0, h, f, T::kDmaA); }
  void read_b(int h, int f) { read(1, h, f, T::kDmaB); }
  void turn(int d) { slot += d; }
  void mfma(int i, int j, int r, int c, int kk) {
    ++g_ops;
    const int t = (int)(mfmas / kPerStep);
    const Read &a = frag[0][i][kk * T::kQM + r], &b = frag[1][j][kk * T::kQN + c];
    if (a.step != t) fail("an MFMA takes another step's rows of x", 0, i);
    if (b.step != t) fail("an MFMA takes another step's rows of W", 1, j);
    if (!seen.insert({i, j, r, c, kk}).second) fail("a block is multiplied twice", 0, i);
    use(a);
    use(b);
    if (++mfmas % kPerStep == 0) seen.clear();
  }
  template <int N>
  void wait_vm() {
    while (dma.size() > (size_t)N) {
      if (++dma.front()->landed == dma.front()->issued) dma.front()->landed_epoch = epoch;
      dma.pop_front();
    }
  }
  template <int N>
  void wait_lgkm() {
    end_reads(N);
  }
  void barrier() { ++epoch; }
  void fence() {}
};

// n steps, run in `parts` calls (the kernel runs K in four segments for some tiles).
template <class T>
void check(const char* name, int n, int parts) {
  Recorder<T> o;
  o.name = name;
  o.n = n;
  QuadSchedule<T> s;
  s.stage_first(o, n);
  s.read_first(o);
  for (int k = 1; k <= parts; ++k) s.steps(o, n, k * n / parts);
  if (o.mfmas != n * Recorder<T>::kPerStep) {
    std::printf("%s, %d steps: %ld MFMAs\n", name, n, o.mfmas);
    std::exit(1);
  }
}
template <class T>
void check_all(const char* name) {
  for (int n = 1; n <= 4 * T::kRing + 3; ++n)
    for (int parts : {1, 4}) check<T>(name, n, parts);
}
}  // namespace

int main() {
  check_all<TileL>("256 x 256");
  check_all<TileP>("192 x 256");
  check_all<TileQ>("256 x 192");
  check_all<TileH>("256 x 128");
  check_all<TileM>("128 x 128");
  std::printf("%ld operations\n", g_ops);
}
