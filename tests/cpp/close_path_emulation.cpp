// The search for the closed path (csrc/close_path.hpp) on the CPU: a fiber per thread of the workgroup, against the cheapest
// closed path by the plain recursion.  The lanes of a wave that have come to the same wave operation take it together, the
// earliest one in the source first; between two barriers the waves run one after the other, each as far as the barrier, in the
// order given: what a wave reads must not depend on how far the others have come.  A row on its way into LDS is rubbish until it
// is waited for.  (Whoever has left the search meets the others at a barrier before anything else: block_passes.)
//   close_path_emulation KIND THREADS ORDER TILES [SEED]    e.g. gauss 256 3210 8    exit code 0: no fault
// Prints how the searches ended: early settled at the free path's group, step0 settled at step 0, (second: in the second attempt,
// lowered: with a step done again under a lower limit,) refused before the first attempt, full and gave_up unsettled.
#undef _FORTIFY_SOURCE  // whose longjmp refuses to leave a stack for another
#include <immintrin.h>
#include <setjmp.h>
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <random>
#include <string>
#include <vector>

namespace {
constexpr int kThreads = 256, kSteps = 128, kSeq = 256, kGroups = 4096, kLanes = 64;
enum Stop { kRunnable, kFirst, kBallot, kRead, kXor, kBarrier, kEnd };
struct Fiber {
  ucontext_t start;
  jmp_buf at;
  bool started = false;
  std::vector<char> stack;
  Stop stop = kRunnable;
  int line = 0, other = 0;
  uint64_t value = 0;
  struct Load {
    const char* from;
    char* to;
  };
  std::deque<Load> loads;
};
std::vector<Fiber> fibers;
ucontext_t scheduler_start;
jmp_buf scheduler;
int running = 0;

void pause_at(Stop why, int line) {
  const int me = running;
  fibers[me].stop = why, fibers[me].line = line;
  if (!_setjmp(fibers[me].at)) _longjmp(scheduler, 1);
}
void resume(int t) {
  running = t;
  fibers[t].stop = kRunnable;
  if (_setjmp(scheduler)) return;
  if (fibers[t].started) _longjmp(fibers[t].at, 1);
  fibers[t].started = true;
  swapcontext(&scheduler_start, &fibers[t].start);
}
uint64_t wave_op(Stop what, uint64_t v, int other, int line) {
  const int me = running;
  fibers[me].value = v, fibers[me].other = other;
  pause_at(what, line);
  return fibers[me].value;
}
[[noreturn]] void wrong(const char* what) {
  std::printf("%s\n", what);
  std::exit(2);
}

// wave w up to its next barrier or to its end
Stop run_wave(int w, int& line) {
  Fiber* const f = &fibers[size_t(w) * kLanes];
  for (;;) {
    for (int l = 0; l < kLanes; ++l)
      if (f[l].stop == kRunnable) resume(w * kLanes + l);
    int first = -1;
    for (int l = 0; l < kLanes; ++l)
      if (f[l].stop < kBarrier && (first < 0 || f[l].line < f[first].line)) first = l;
    if (first < 0) {
      for (int l = 1; l < kLanes; ++l)
        if (f[l].stop != f[0].stop || f[l].line != f[0].line) wrong("the lanes of a wave stopped at different barriers");
      line = f[0].line;
      return f[0].stop;
    }
    const Stop what = f[first].stop;
    const int at = f[first].line;
    bool in[kLanes];
    uint64_t given[kLanes], mask = 0;
    for (int l = 0; l < kLanes; ++l) {
      in[l] = f[l].stop == what && f[l].line == at;
      given[l] = f[l].value;
      if (in[l]) mask |= uint64_t(given[l] & 1u) << l;
    }
    for (int l = 0; l < kLanes; ++l) {
      if (!in[l]) continue;
      const int from = what == kRead ? f[l].other : what == kXor ? l ^ f[l].other : first;
      if (what != kBallot && !in[from]) wrong("a lane reads one that is not there");
      f[l].value = what == kBallot ? mask : given[from];
      f[l].stop = kRunnable;
    }
  }
}

struct double2 {
  double x, y;
};
struct Smem {
  double E[32 * 64];
  double M[4096];
  float x[kSeq];
  uint16_t st[kSteps];
  uint32_t close_count[2], close_least[2], close_ok;
} sm_all;
struct Unit {
  double pre;
};
constexpr uint32_t kSat = 0xffffffffu, kWinnerMax = kSat - (1u << 20);
uint32_t sat_add(uint32_t a, uint32_t b) { return a + b < a ? kSat : a + b; }
uint32_t owner32(uint32_t jj) {
  const uint32_t c = jj >> 4;
  return (c >> 2) | ((c & 3u) << 5) | (((jj >> 3) & 1u) << 7);
}
int opaque_tid() { return running & (kThreads - 1); }
int opaque_tid_wide() { return running; }
float fp16_value(uint16_t bits) { return _cvtsh_ss(bits); }

char* lds(uint32_t at) { return reinterpret_cast<char*>(&sm_all) + at; }
template <class T>
T get(uint32_t at) {
  T v;
  std::memcpy(&v, lds(at), sizeof v);
  return v;
}
template <class T>
void put(uint32_t at, T v) {
  std::memcpy(lds(at), &v, sizeof v);
}
uint32_t lds_at(const void* p) { return uint32_t(static_cast<const char*>(p) - lds(0)); }
unsigned long long lds_min(uint32_t at, unsigned long long v) {
  const auto old = get<unsigned long long>(at);
  if (v < old) put(at, v);
  return old;
}
uint32_t lds_add(uint32_t at, uint32_t v) {
  const auto old = get<uint32_t>(at);
  put(at, old + v);
  return old;
}
void lds_min(uint32_t at, uint32_t v) {
  if (v < get<uint32_t>(at)) put(at, v);
}
int rounds = 0, steps_done = 0, last_step = 0, attempts = 0;  // of thread 0's search
uint32_t list0_at = 0;
void lds_put32(uint32_t at, uint32_t v) { put(at, v); }
void lds_put64(uint32_t at, unsigned long long v) { put(at, v); }
void lds_put16(uint32_t at, uint32_t v) {
  put(at, uint16_t(v));
  if (steps_done++ == 0) list0_at = at - 2 * (kSteps - 1);  // the search's first step is the sequence's last
  last_step = int(at - list0_at) / 2;
  if (last_step == kSteps - 1) ++attempts;
}
uint32_t lds_get16(uint32_t at) { return get<uint16_t>(at); }
void lds_get_32_64(uint32_t at32, uint32_t at64, uint32_t& v32, unsigned long long& v64) {
  v32 = get<uint32_t>(at32), v64 = get<unsigned long long>(at64);
  if (running == 0) ++rounds;
}
void load_row(const char* from, uint32_t lane, char* to) {
  std::memset(to + 16 * lane, 0xa5, 16);
  fibers[size_t(running)].loads.push_back({from + 16 * lane, to + 16 * lane});
}
void wait_lds() {}
template <size_t kLeft>
void wait_loads() {
  auto& q = fibers[size_t(running)].loads;
  for (; q.size() > kLeft; q.pop_front()) std::memcpy(q.front().to, q.front().from, 16);
}
uint32_t units_of(double q) { return !(q > 0) ? 0 : q >= 4294967295.0 ? kSat : uint32_t(q); }
uint32_t mbcnt_lo(uint32_t mask, uint32_t v) {
  const int l = running & 63;
  return v + uint32_t(__builtin_popcount(l >= 32 ? mask : mask & ((1u << l) - 1u)));
}
uint32_t mbcnt_hi(uint32_t mask, uint32_t v) {
  const int l = running & 63;
  return v + (l < 32 ? 0u : uint32_t(__builtin_popcount(mask & ((1u << (l - 32)) - 1u))));
}
uint32_t umul24(uint32_t a, uint32_t b) { return (a & 0xffffffu) * (b & 0xffffffu); }
int hi_word(double v) { return int(__builtin_bit_cast(uint64_t, v) >> 32); }
int lo_word(double v) { return int(uint32_t(__builtin_bit_cast(uint64_t, v))); }
double from_words(int hi, int lo) { return __builtin_bit_cast(double, uint64_t(uint32_t(hi)) << 32 | uint32_t(lo)); }
using std::max;
using std::min;

#define __device__
#define __forceinline__ inline
#define __restrict__
#define __hip_atomic_load(p, order, scope) (*(p))
#define __umul24(a, b) umul24(a, b)
#define __double2hiint(v) hi_word(v)
#define __double2loint(v) lo_word(v)
#define __hiloint2double(h, l) from_words(h, l)
#define __builtin_amdgcn_readfirstlane(v) int(wave_op(kFirst, uint32_t(v), 0, __LINE__))
#define __builtin_amdgcn_readlane(v, lane) int(wave_op(kRead, uint32_t(v), lane, __LINE__))
#define __builtin_amdgcn_ballot_w64(v) wave_op(kBallot, v, 0, __LINE__)
#define __builtin_amdgcn_mbcnt_lo(m, v) mbcnt_lo(m, v)
#define __builtin_amdgcn_mbcnt_hi(m, v) mbcnt_hi(m, v)
#define __shfl_xor(v, o, width) wave_op(kXor, v, o, __LINE__)
#define __builtin_amdgcn_s_barrier() pause_at(kBarrier, __LINE__)
#define __syncthreads() pause_at(kBarrier, __LINE__)
#include "../../behemoth-qtip_amd/csrc/close_path.hpp"

// ---- the tile: codebook, inputs, the free pass with its bounds, the closed path by the plain recursion
uint32_t book[512];
struct Tile {
  double x[kSeq];
  Unit unit;
  uint32_t ov, winner, grown;
  bool settled;  // the free pass's decisions are all clear
  uint16_t free_path[kSteps], closed[kSteps];
  std::vector<char> slot;
} tile;
constexpr uint32_t kMargin = 160;

void errors(int t, std::vector<uint32_t>& e) {
  for (int i = 0; i < 1024; ++i) {
    const uint32_t w = book[i & 511];
    const double l0 = fp16_value(uint16_t(w)), l1 = fp16_value(uint16_t(w >> 16)), pre = tile.unit.pre;
    const double a = (i >> 9 ? -l0 : l0) * pre - tile.x[t] * pre, b = l1 * pre - tile.x[t + 1] * pre;
    e[size_t(i)] = units_of(std::fma(a, a, std::fma(b, b, 0.5)));
  }
}
uint32_t entry_of(uint32_t s) { return ((s * (s + 1u)) >> 6) & 1023u; }
// one step of the recursion; `from` may hold a saturated or 64-bit metric
template <class T, class Add>
void forward(const std::vector<T>& from, const std::vector<uint32_t>& e, std::vector<T>& to, Add add) {
  for (uint32_t j = 0; j < uint32_t(kGroups); ++j) {
    T best = ~T(0);
    for (uint32_t d = 0; d < 16; ++d) {
      const uint32_t s = d << 12 | j;
      best = min(best, add(from[s >> 4], e[entry_of(s)]));
    }
    to[j] = best;
  }
}
void free_pass() {
  std::vector<uint32_t> e(1024);
  std::vector<std::vector<uint32_t>> M(kSteps + kTurn + 1, std::vector<uint32_t>(kGroups)), err(kSteps + kTurn);
  for (int i = 0; i < kSteps + kTurn; ++i) {
    errors((2 * i + kSeq / 2) & (kSeq - 1), e);
    err[size_t(i)] = e;
    forward(M[size_t(i)], e, M[size_t(i) + 1], sat_add);
  }
  uint16_t* const bounds = reinterpret_cast<uint16_t*>(tile.slot.data() + kBoundsAt);
  tile.grown = kSat;
  for (int i = 1; i <= kSteps + kTurn; ++i)
    for (uint32_t j = 0; j < uint32_t(kBoundRow); ++j)
      bounds[size_t(i) * kBoundRow + owner32(j) * 8 + (j & 7u)] = uint16_t(M[size_t(i)][j] >> 16);
  for (int j = 0; j < kBoundRow; ++j) {
    const uint32_t now = M[kSteps + kTurn][size_t(j)] >> 16, before = M[kTurn][size_t(j)] >> 16;
    tile.grown = min(tile.grown, now > before ? now - before - 1u : 0u);
  }
  tile.grown <<= 16;
  uint32_t best = 0, second = kSat;
  for (uint32_t j = 1; j < uint32_t(kBoundRow); ++j) {
    if (M[kSteps][j] < M[kSteps][best]) second = M[kSteps][best], best = j;
    else second = min(second, M[kSteps][j]);
  }
  tile.winner = M[kSteps][best];
  tile.settled = second - tile.winner >= kMargin && tile.winner < kWinnerMax;
  uint32_t g = best;
  for (int i = kSteps - 1; i >= kSteps / 2; --i) {
    uint32_t c1 = kSat, c2 = kSat, s1 = 0;
    for (uint32_t d = 0; d < 16; ++d) {
      const uint32_t s = d << 12 | g, c = sat_add(M[size_t(i)][s >> 4], err[size_t(i)][entry_of(s)]);
      if (c < c1) c2 = c1, c1 = c, s1 = s;
      else c2 = min(c2, c);
    }
    tile.settled = tile.settled && c2 - c1 >= kMargin;
    tile.free_path[i] = uint16_t(s1), g = s1 >> 4;
  }
  tile.ov = g;
}
void closed_path() {
  std::vector<uint32_t> e(1024);
  std::vector<std::vector<uint64_t>> D(kSteps + 1, std::vector<uint64_t>(kGroups, uint64_t(1) << 60));
  std::vector<std::vector<uint32_t>> err(kSteps);
  D[0][tile.ov] = 0;
  for (int p = 0; p < kSteps; ++p) {
    errors(2 * p, e);
    err[size_t(p)] = e;
    forward(D[size_t(p)], e, D[size_t(p) + 1], [](uint64_t a, uint32_t b) { return a + b; });
  }
  uint32_t g = tile.ov;
  for (int p = kSteps - 1; p >= 0; --p) {
    uint64_t c1 = ~0ull;
    uint32_t s1 = 0;
    for (uint32_t d = 0; d < 16; ++d) {
      const uint32_t s = d << 12 | g;
      const uint64_t c = D[size_t(p)][s >> 4] + err[size_t(p)][entry_of(s)];
      if (c < c1) c1 = c, s1 = s;
    }
    tile.closed[p] = uint16_t(s1), g = s1 >> 4;
  }
}

int threads = kThreads;
bool answers[2 * kThreads];
void thread_main() {
  const int me = running;
  const uint32_t* const hist = reinterpret_cast<const uint32_t*>(tile.slot.data());
  answers[me] = threads == kThreads
                    ? close_path<false>(sm_all, book, hist, tile.ov, tile.winner, tile.grown, kMargin, tile.unit)
                    : close_path<true>(sm_all, book, hist, tile.ov, tile.winner, tile.grown, kMargin, tile.unit);
  pause_at(kBarrier, 0);
  pause_at(kEnd, 0);
}

// a codebook value, an input: fp16 values
double as_fp16(double v) { return _cvtsh_ss(_cvtss_sh(float(v), 0)); }
void make_tile(const std::string& kind, std::mt19937_64& gen) {
  std::normal_distribution<double> normal;
  std::vector<double> x(kSeq);
  for (double& v : x) v = 0.9 * normal(gen);
  int unit_log2 = 20;
  if (kind == "join") {  // large values around the place where the closed path's ends meet
    for (int t = 0; t < 12; ++t) x[size_t(t)] *= 4.0, x[size_t(kSeq - 1 - t)] *= 4.0;
  } else if (kind == "flat") {  // many paths of nearly the same cost
    for (double& v : x) v *= 0.02;
  } else if (kind == "alike") {  // the same values again and again
    for (int t = 8; t < kSeq; ++t) x[size_t(t)] = x[size_t(t & 7)];
  } else if (kind == "mirror") {  // decoded values of a path that arrives at the complement of its start
    uint32_t s = uint32_t(gen()) & 0xffffu;
    const uint32_t s0 = s;
    for (int p = 0; p < kSteps; ++p) {
      if (p > 0) s = (s << 4 | (p < kSteps - 3 ? uint32_t(gen()) & 15u : (65535u - s0) >> 4 * (kSteps - p) & 15u)) & 0xffffu;
      const uint32_t e = entry_of(s), w = book[e & 511];
      const double l0 = fp16_value(uint16_t(w)), l1 = fp16_value(uint16_t(w >> 16));
      x[size_t(2 * p)] = (e >> 9 ? -l0 : l0) + 0.02 * x[size_t(2 * p)], x[size_t(2 * p) + 1] = l1 + 0.02 * x[size_t(2 * p) + 1];
    }
  } else if (kind == "coarse") {  // a winner so near the end of the range that the search's limit lies beyond it
    for (double& v : x) v *= 1.0 + 2.0 * double(gen() >> 11) * 0x1p-53;
  } else if (kind != "gauss") {
    wrong("unknown kind");
  }
  for (int t = 0; t < kSeq; ++t) tile.x[t] = as_fp16(x[size_t(t)]);
  // the finest unit that the winner fits with as much room again, which is what the passes aim at; coarse: that it just fits
  const uint32_t enough = kind == "coarse" ? (1u << 30) - (1u << 20) : 1u << 29;
  tile.unit = Unit{std::ldexp(1.0, unit_log2 / 2)};
  free_pass();
  while (unit_log2 < 30 && tile.winner < enough) {
    unit_log2 += 2;
    tile.unit = Unit{std::ldexp(1.0, unit_log2 / 2)};
    free_pass();
  }
}
}  // namespace

int main(int argc, char** argv) {
  if (argc < 5) return 2;
  threads = std::atoi(argv[2]);
  const std::string order = argv[3];
  const int waves = threads / kLanes, tiles = std::atoi(argv[4]);
  if ((threads != kThreads && threads != 2 * kThreads) || int(order.size()) != waves) return 2;
  std::mt19937_64 gen(argc > 5 ? std::strtoull(argv[5], nullptr, 10) : 1);
  std::normal_distribution<double> normal;
  for (uint32_t& w : book) {
    const uint32_t a = _cvtss_sh(float(normal(gen)), 0), b = _cvtss_sh(float(normal(gen)), 0);
    w = a | b << 16;
  }
  tile.slot.resize(kBoundsAt + size_t(kSteps + kTurn + 1) * kBoundRow * 2);
  fibers.resize(size_t(threads));
  for (Fiber& f : fibers) f.stack.resize(1 << 16);
  int early = 0, step0 = 0, second = 0, lowered = 0, refused = 0, full = 0, gave_up = 0, unclear = 0, faults = 0;
  for (int n = 0; n < tiles; ++n) {
    make_tile(argv[1], gen);
    if (!tile.settled) {
      ++unclear;
      continue;
    }
    closed_path();
    std::memset(&sm_all, 0x5a, sizeof sm_all);
    for (int t = 0; t < kSeq; ++t) sm_all.x[t] = float(tile.x[t]);
    std::memcpy(sm_all.st + kSteps / 2, tile.free_path + kSteps / 2, kSteps);
    rounds = steps_done = last_step = attempts = 0;
    for (Fiber& f : fibers) {
      f.started = false, f.stop = kRunnable, f.loads.clear();
      getcontext(&f.start);
      f.start.uc_stack.ss_sp = f.stack.data();
      f.start.uc_stack.ss_size = f.stack.size();
      f.start.uc_link = nullptr;  // a fiber stays where it ends
      makecontext(&f.start, thread_main, 0);
    }
    for (Stop all = kBarrier; all != kEnd;) {
      int line = 0;
      for (int k = 0; k < waves; ++k) {
        int at = 0;
        const int w = order[size_t(k)] - '0';
        const Stop why = run_wave(w, at);
        if (k > 0 && (why != all || at != line)) wrong("the waves stopped at different barriers");
        all = why, line = at;
        if (why == kBarrier)
          for (int l = 0; l < kLanes; ++l) fibers[size_t(w * kLanes + l)].stop = kRunnable;
      }
    }
    for (int t = 1; t < threads; ++t)
      if (answers[t] != answers[0]) wrong("the threads' answers differ");
    for (const Fiber& f : fibers)
      if (!f.loads.empty()) wrong("a load is still on its way at the end");
    if (answers[0]) {
      if (std::memcmp(sm_all.st, tile.closed, sizeof tile.closed)) std::printf("tile %d: states differ\n", n), ++faults;
      if (last_step > 0) ++early;
      else ++step0;
      second += attempts > 1;
    } else {
      if (attempts == 0 && rounds == 0) ++refused;
      else if (rounds == steps_done) ++full;  // every step fitted, the room for all of them ended
      else ++gave_up;
    }
    lowered += answers[0] && rounds > steps_done;
  }
  std::printf("early %d step0 %d second %d lowered %d refused %d full %d gave_up %d unclear %d faults %d\n", early, step0, second,
              lowered, refused, full, gave_up, unclear, faults);
  return faults ? 1 : 0;
}
