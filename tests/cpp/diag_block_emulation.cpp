// The diagonal-block factorization of the device LDL (csrc/ldl_diag.hpp) on the CPU: 256 fibers, one per thread of the
// workgroup, against the host's factorization of the same block (csrc/host_ldl_diag.cpp), bit for bit.
// The 64 fibers of a wave meet at every lane read; between two barriers of the workgroup the waves run one after the
// other, each as far as the barrier, in an order given on the command line: what a wave reads before a barrier must not
// depend on how far the others have come.
//   diag_block_emulation KB ORDER [SEED]     e.g. 256 3210      exit code 0: every word equal
#undef _FORTIFY_SOURCE  // whose longjmp refuses to leave a stack for another
#include <setjmp.h>
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

namespace {
constexpr int kLanes = 64, kWaves = 4, kThreads = kLanes * kWaves;
enum Stop { kLaneRead, kBarrier, kEnd };
// (a fiber is started on its stack by swapcontext; from then on the switches are jumps, which need no system call)
struct Fiber {
  ucontext_t start;
  jmp_buf at;
  bool started = false;
  std::vector<char> stack;
  Stop stop = kLaneRead;
  int published[2] = {0, 0};  // of this lane read and the one before it: a lane may be one ahead of the others
  int turn = 0;
};
Fiber fibers[kThreads];
ucontext_t scheduler_start;
jmp_buf scheduler;
int running = 0;

void pause_at(Stop why) {
  const int me = running;
  fibers[me].stop = why;
  if (!_setjmp(fibers[me].at)) _longjmp(scheduler, 1);
}
void resume(int t) {
  running = t;
  if (_setjmp(scheduler)) return;
  if (fibers[t].started) _longjmp(fibers[t].at, 1);
  fibers[t].started = true;
  swapcontext(&scheduler_start, &fibers[t].start);
}
int read_lane(int v, int lane) {
  const int me = running, turn = fibers[me].turn;
  fibers[me].published[turn] = v;
  fibers[me].turn = turn ^ 1;
  pause_at(kLaneRead);
  return fibers[me / kLanes * kLanes + lane].published[turn];
}
struct ThreadIdx {
  struct X {
    operator int() const { return running; }
  } x;
} threadIdx;
struct double2 {
  double x, y;
};
double2 make_double2(double x, double y) { return {x, y}; }
}  // namespace

#define __device__
#define __forceinline__ inline
#define __restrict__
#define __builtin_amdgcn_readlane(v, lane) read_lane(v, lane)
#define __builtin_amdgcn_readfirstlane(v) read_lane(v, 0)
#define __builtin_amdgcn_sched_barrier(mask) ((void)0)
#define __syncthreads() pause_at(kBarrier)
#include "../../behemoth-qtip_amd/csrc/ldl_diag.hpp"

namespace qtipmi {
bool factor_diag_avx2(double* A, long ld, int kb, double* T, int ldt);
}

namespace {
struct Call {
  double* A;
  long ld;
  int kb;
  double *rdiag, *inv;
  int* bad;
} call;
alignas(16) qtipmi::DiagLds lds;

void thread_main() {
  qtipmi::factor_diag_block(lds, call.A, call.ld, call.kb, call.rdiag, call.inv, call.bad);
  pause_at(kEnd);
}

// wave w up to its next barrier, or to its end
Stop run_wave(int w) {
  for (;;) {
    for (int l = 0; l < kLanes; ++l) resume(w * kLanes + l);
    const Stop why = fibers[w * kLanes].stop;
    for (int l = 1; l < kLanes; ++l)
      if (fibers[w * kLanes + l].stop != why) {
        std::printf("the lanes of wave %d stopped at different places\n", w);
        std::exit(2);
      }
    if (why != kLaneRead) return why;
  }
}
}  // namespace

int main(int argc, char** argv) {
  if (argc < 3 || std::strlen(argv[2]) != kWaves) return 2;
  const int kb = std::atoi(argv[1]), rows = 2 * kb;
  const long ld = kb + 16;
  std::mt19937_64 gen(argc > 3 ? std::strtoull(argv[3], nullptr, 10) : 1);
  std::normal_distribution<double> normal;
  std::vector<double> X(size_t(rows) * kb), A(size_t(kb) * ld, 0.0), rdiag(kb), inv(size_t(kb) * 16);
  for (double& v : X) v = normal(gen);
  for (int i = 0; i < kb; ++i)
    for (int j = 0; j <= i; ++j) {
      double s = 0;
      for (int r = 0; r < rows; ++r) s += X[size_t(r) * kb + i] * X[size_t(r) * kb + j];
      A[i * ld + j] = s / rows;
    }
  std::vector<double> want = A;
  const int ldt = (kb + 31) / 32 * 32;
  std::vector<double> T(size_t(kb) * ldt);
  if (!qtipmi::factor_diag_avx2(want.data(), ld, kb, T.data(), ldt)) return 2;

  int bad = 0;
  call = {A.data(), ld, kb, rdiag.data(), inv.data(), &bad};
  for (Fiber& f : fibers) {
    f.stack.resize(1 << 16);
    getcontext(&f.start);
    f.start.uc_stack.ss_sp = f.stack.data();
    f.start.uc_stack.ss_size = f.stack.size();
    f.start.uc_link = nullptr;  // a fiber stays where it ends
    makecontext(&f.start, thread_main, 0);
  }
  for (Stop all = kBarrier; all != kEnd;) {
    for (int k = 0; k < kWaves; ++k) {
      const Stop why = run_wave(argv[2][k] - '0');
      if (k > 0 && why != all) {
        std::printf("the waves stopped at different barriers\n");
        return 2;
      }
      all = why;
    }
  }
  long differ = 0;
  for (int i = 0; i < kb; ++i) {
    for (int j = 0; j <= i; ++j) differ += std::memcmp(&A[i * ld + j], &want[i * ld + j], sizeof(double)) != 0;
    const double r = 1.0 / want[i * ld + i];
    differ += std::memcmp(&rdiag[i], &r, sizeof r) != 0;
  }
  std::printf("kb %d, waves in the order %s: %ld words differ, flag %d\n", kb, argv[2], differ, bad);
  return differ || bad ? 1 : 0;
}
