// The second pass of a tile as a search (viterbi.hip): close_path, in a file of its own so that
// tests/cpp/close_path_emulation.cpp can run it on the CPU, its waves in any order between two barriers.
// Included inside viterbi.hip's namespace.  What it takes from there: kThreads, kSteps, kGroups, Smem, Unit, kSat, kWinnerMax,
// sat_add, owner32, opaque_tid(_wide), fp16_value, and the operations that have a form of their own on the device (lds_at and the
// lds_ functions, units_of, load_row, wait_lds, wait_loads).
#pragma once

// What the search for the closed path needs of a free pass (close_path below) lies behind the 32-bit kept metrics: the
// upper halves of the metrics entering the steps 1 .. 128 + kTurn (kBoundRow values each).
constexpr int kTurn = 48;              // steps the free pass runs on into the sequence's second round
constexpr int kBoundRow = kGroups / 2;
constexpr int kCloseList = 256;        // room for the partial paths of a step
constexpr int kCloseSlots = 512;       // hash slots in which partial paths of one group meet
constexpr int kClosePaths = 3520;      // partial paths of all steps together
constexpr int kCloseRing = 4;          // rows of bounds in LDS
constexpr size_t kBoundsAt = size_t(64) * kGroups * sizeof(uint32_t);                       // bytes into the slot
static_assert(kTurn % 2 == 0 && kTurn < kSteps / 2);

// The tail-biting pass without its forward recursion.  The cheapest path from group ov before step 0 back to ov after step
// 127 is searched for from its end, step 127 down to step 0: of the partial paths (a group entering a step and the
// cheapest completion from there to ov) only those are followed that can still belong to a closed path under a limit, and
// the free pass of the same block says which.  It ran on the same values rotated by half the sequence and then kTurn steps
// into its second round, so with M_i its metrics entering its step i, a path from ov at the sequence's start to group h
// entering step p costs at least
//     M_{64 + p}[h] - M_64[ov]              for p <= 64 + kTurn  (M_{64 + p}[h] is at most M_64[ov] + that cost), and
//     M_{p - 64}[h] + grown - M_64[ov]      beyond, `grown` being the least growth of a metric over one round
// (the recursion is monotone and commutes with adding a constant).  The free path itself goes through ov, and a closed path
// differs from it around the join only, by 0.2 to 1.2 of a cost of 14 (normalized weights), most of which lies in the
// kTurn steps behind the join that the bounds have seen: the search follows 1 to 20 partial paths a step where the
// forward recursion updates 4096 groups from 65536 candidates.
// What is left to pay is often the mirror: free paths come in complementary pairs, the metrics do not say which of the two
// a group belongs to, and the closed path through ov must not arrive at its complement.  Half of the tiles have to
// change over somewhere, at a cost of up to 0.25.  The others are done as soon as the free path's own group is the only
// one left near the limit: the rest of the free path leads from it to ov, at the least cost there is.
// Costs are the 32-bit passes' integers in the free pass's unit, summed exactly; bounds are kept as the upper halves of
// the metrics, which makes them weaker by less than 65536 units and never too large.  A result counts if it is under the
// limit the search ended with (a path left out then costs more) and no two paths that met in a group were closer than
// `margin`: the winner then beats every other closed path by that much, and the fp64 recursion takes it.  Otherwise
// the search is tried once more with a higher limit, then false is returned and the caller runs the pass.
// What bounds it: latency.  A step is a chain of five LDS round trips and some 150 instructions, 0.85 us by itself and
// 1.1 us beside two other workgroups, 120 steps a tile; the pipes it leaves idle are the other workgroups' forward passes'.
// Per block with three workgroups on a compute unit (LDLQ of 768 tile rows) 134 us instead of 268 + 76 for the forward
// recursion and its trace-back, with 20 us more in the free pass and its trace-back; 99.7 % of the searches settle their block.
// (768 tile rows through 128 blocks 89.3 -> 69.9 ms; kTurn 40 / 48 / 56: 70.0 / 69.9 / 71.3; at most 48 / 64 / 128 partial
// paths in the first attempt: 70.6 / 70.0 / 70.7, three attempts with up to 256: 73.3, one: 73.8.)
template <bool kWide>
__device__ __forceinline__ bool close_path(Smem& sm, const uint32_t* tl, const uint32_t* __restrict__ hist32, uint32_t ov,
                                           uint32_t winner, uint32_t grown, uint32_t margin, const Unit unit) {
  constexpr uint32_t kT = kWide ? 2 * kThreads : kThreads;
  typedef unsigned long long u64;
  const uint32_t tid = uint32_t(kWide ? opaque_tid_wide() : opaque_tid()), lane = tid & 63u, d = tid & 15u;
  const int wave = __builtin_amdgcn_readfirstlane(int(tid) >> 6);
  const char* const bounds = reinterpret_cast<const char*>(hist32) + kBoundsAt;
  // LDS: a ring of rows of bounds in sm.E; in sm.M the codebook's 512 entries and the inputs as pairs of fp64 values times
  // Unit::pre, the meeting places, two lists of partial paths (cost << 32 | place bits << 20 | position of the path
  // continued in its step's list << 12 | group) and the lower words of all of them in the order found
  char* const area = reinterpret_cast<char*>(sm.M);
  double2* const book = reinterpret_cast<double2*>(area);
  double2* const input = book + 512;
  u64* const meet = reinterpret_cast<u64*>(input + kSteps);
  u64* const lists = meet + kCloseSlots;
  uint32_t* const paths = reinterpret_cast<uint32_t*>(lists + 2 * kCloseList);
  uint16_t* const list0 = reinterpret_cast<uint16_t*>(paths + kClosePaths);  // where the paths of a step begin there
  static_assert(kCloseRing * kBoundRow * 2 <= sizeof(sm.E) &&
                (512 + kSteps) * 16 + (kCloseSlots + 2 * kCloseList) * 8 + kClosePaths * 4 + kSteps * 2 <= sizeof(sm.M));
  // Byte offset of group h in a row: bits 4..11 of h and 0..3 of its digit d apart.  Group h = (d << 8) | (j >> 4) of a
  // partial path to group j lies at the place of h or, from 2048 up, of 4095 - h = ~h, so bits and digit contribute by XOR.
  auto place = [](uint32_t jj) -> uint32_t { return (owner32(jj) * 8u + (jj & 7u)) * 2u; };
  const uint32_t d_place = d < 8u ? place(d << 8) : place(((15u - d) << 8) | 0xffu);
  const uint32_t d_meet = lds_at(meet);
  const uint32_t d_slot = ((d & 1u) << 8 | (d >> 1) << 5) * 8u;
  const uint32_t d_next = place(d << 4) << 20;  // what the digit adds to the place bits of the group it leads to
  auto issue = [&](int p) {  // the bounds of step p, 1 KB per wave of the first four
    const int r = p <= kSteps / 2 + kTurn ? p + kSteps / 2 : p - kSteps / 2;
    if (wave < 4)
      load_row(bounds + size_t(r) * (kBoundRow * 2) + wave * 1024, lane,
               reinterpret_cast<char*>(sm.E) + uint32_t(p) % kCloseRing * (kBoundRow * 2) + wave * 1024);
  };
  auto lds_barrier = [] {  // orders LDS, not the loads in flight
    wait_lds();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  const uint32_t ov_low = ov < 2048u ? ov : 4095u - ov;
  // M_64[ov], rounded down: what every bound above starts from
  const uint32_t start = uint32_t(__builtin_amdgcn_readfirstlane(int(__hip_atomic_load(
      reinterpret_cast<const uint16_t*>(bounds + size_t(kSteps / 2) * (kBoundRow * 2) + place(ov_low)), __ATOMIC_RELAXED,
      __HIP_MEMORY_SCOPE_WORKGROUP)))) << 16;
  const uint32_t least = uint32_t(__builtin_amdgcn_readfirstlane(int(sat_add(start, grown))));
  __syncthreads();
  for (uint32_t g = tid; g < kCloseSlots; g += kT) meet[g] = ~0ull;
  for (uint32_t g = tid; g < 512u; g += kT) {
    const uint32_t w = tl[g];
    book[g].x = double(fp16_value(uint16_t(w))) * unit.pre;
    book[g].y = double(fp16_value(uint16_t(w >> 16))) * unit.pre;
  }
  if (tid < kSteps) input[tid].x = double(sm.x[2 * tid]) * unit.pre, input[tid].y = double(sm.x[2 * tid + 1]) * unit.pre;
  const u64 root = (place(ov >> 4) << 20) | ov;
  if (tid < 2) sm.close_count[tid] = 0, sm.close_least[tid] = kSat;
  // turn: one round of the loop below, a step or another try at it with a lower limit; the stamp, counted downwards in the
  // keys, tells the meeting places' entries of different turns apart.  Two counters, used in turn, run on; `seen` is what
  // the one in use stood at.
  uint32_t stamp = 0xfffff000u, counter = lds_at(sm.close_count), seen = 0, seen_other = 0;
  bool ok = false;
#pragma nounroll
  for (int attempt = 0; attempt < 2 && !ok; ++attempt) {
    uint32_t limit = least + 131072u + winner / (attempt ? 20u : 32u);
    const uint32_t cap = attempt ? 128u : 64u;  // partial paths of a step
    if (limit >= kWinnerMax || limit < least) return false;
    issue(kSteps - 1);
    issue(kSteps - 2);
    issue(kSteps - 3);
    issue(kSteps - 4);
    wait_loads<3>();
    lds_barrier();
    uint32_t n = 1, total = 0, found = 0;  // the present list's length; all paths so far
    int p = kSteps - 1;
    double2 x = input[p];
    u64 first = root;
#pragma nounroll
    for (;;) {
      const u64* const list = lists + (p & 1 ? 0 : kCloseList);
      const uint32_t next = lds_at(lists + (p & 1 ? kCloseList : 0));
      const uint32_t row = lds_at(sm.E) + uint32_t(p) % kCloseRing * (kBoundRow * 2);
      const uint32_t most = limit - (p > kSteps / 2 + kTurn ? grown : 0u);
      // every fourth step of the first half the free path's group is looked at by itself, and at the end of the second
      // round's steps the smallest bound
      const bool on_free = p < kSteps / 2 && (p & 3) == 0, watched = on_free || p == kSteps / 2 + kTurn;
      uint32_t on_path = kSat;
      if (on_free) on_path = uint32_t(__builtin_amdgcn_readfirstlane(int(sm.st[kSteps / 2 + p]))) >> 4;
      u64 path = first;
      for (uint32_t k = tid >> 4; k < n; k += kT / 16) {
        if (k >= kT / 16) path = list[k];
        const uint32_t lo = uint32_t(path), s = (d << 12) | (lo & 0xfffu), h = s >> 4;
        const uint32_t v = __umul24(s, s) + s;
        const double2 l = book[(v >> 6) & 511u];
        const uint32_t bound = lds_get16(row + ((lo >> 20) ^ d_place));
        const double lx = __hiloint2double(__double2hiint(l.x) ^ int((v << 16) & 0x80000000u), __double2loint(l.x));
        const double a0 = lx - x.x, a1 = l.y - x.y;
        const uint32_t err = units_of(__builtin_fma(a0, a0, __builtin_fma(a1, a1, 0.5)));
        const uint32_t c = sat_add(uint32_t(path >> 32), err), f = sat_add(bound << 16, c);
        if (f <= most) {
          bool keep = true;
          uint32_t doubt = 0;
          if (n > 1) {  // (the sixteen continuations of one path lead to sixteen groups)
            const u64 old = lds_min(d_meet + (((lo >> 1) & 0x7f8u) ^ d_slot), (u64(stamp | (c >> 20)) << 32) | ((c << 12) | h));
            if (uint32_t(old >> 32) < stamp + 4096u && (uint32_t(old) & 0xfffu) == h) {  // another path to h
              const uint32_t o = uint32_t(old >> 12);
              keep = c < o;
              doubt = min(o - c, c - o) < margin ? 0x10000u : 0u;  // counted as more than any list holds
            }
          }
          if (watched) lds_min(lds_at(sm.close_least) + (h == on_path ? 4u : 0u), f);
          if (doubt) (void)lds_add(counter, doubt);
          if (keep) {
            const u64 mask = __builtin_amdgcn_ballot_w64(true);
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
            uint32_t at = 0;
            if (rank == 0) at = lds_add(counter, uint32_t(__builtin_popcountll(mask)));
            at = uint32_t(__builtin_amdgcn_readfirstlane(int(at))) - seen + rank;
            if (at < kCloseList) {
              const uint32_t word = d_next | (lo & 0x700u) << 13 | (lo & 0x800u) << 20 | k << 12 | h;
              lds_put64(next + 8u * at, (u64(c) << 32) | word);
              lds_put32(lds_at(paths + total) + 4u * at, word);
            }
          }
        }
      }
      // the next step's inputs and bounds (the two rows after them may be under way)
      const double2 x_next = input[p > 0 ? p - 1 : 0];
      if (p >= 3) wait_loads<2>();
      else wait_loads<0>();
      lds_barrier();
      uint32_t count;
      u64 path_next;
      lds_get_32_64(counter, next + 8u * (tid >> 4), count, path_next);
      count = uint32_t(__builtin_amdgcn_readfirstlane(int(count)));
      const uint32_t m = count - seen;
      seen = seen_other, seen_other = count, counter ^= lds_at(sm.close_count) ^ lds_at(sm.close_count + 1), stamp -= 4096u;
      if (m - 1u >= cap) {
        // none left, or two too close together, or too many: those once more with a lower limit
        if (m == 0 || m >= 0x10000u || limit - least < 4096u || stamp < 0x10000000u) break;
        limit -= (limit - least) / 4;
        if (watched) {
          lds_barrier();
          if (tid < 2) lds_put32(lds_at(sm.close_least + tid), kSat);
          lds_barrier();
        }
        continue;
      }
      if (tid == 0) lds_put16(lds_at(list0 + p), total);
      if (watched) {
        const uint32_t off = uint32_t(__builtin_amdgcn_readfirstlane(int(sm.close_least[0])));
        const uint32_t on = uint32_t(__builtin_amdgcn_readfirstlane(int(sm.close_least[1])));
        if (on_free && on < kWinnerMax && on + 131072u + margin <= off && on + 65536u + margin <= limit) {
          found = m;
          break;
        }
        // a path that has come to the free path's group is closed by it, at a cost below on + 131072 - M_64[ov]
        if (on < kWinnerMax) limit = min(limit, on + 131072u + 2u * min(margin, 1u << 20));
        if (!on_free) limit = min(limit, off + min(kSat - off, 131072u + winner / (attempt ? 32u : 56u)));
        lds_barrier();
        if (tid < 2) lds_put32(lds_at(sm.close_least + tid), kSat);
      }
      if (p == 0) {
        found = m;
        break;
      }
      total += m;
      if (total + kCloseList > kClosePaths) break;
      n = m;
      --p;
      if (p >= 3) issue(p - 3);  // into the buffer of step p + 1
      first = path_next, x = x_next;
    }
    wait_loads<0>();
    __syncthreads();
    if (tid < 2) sm.close_least[tid] = kSat;
    // The verdict is the first wave's, and the others hear it behind the barrier: a search that ends on the free path writes
    // the states over that path's own, which only that wave may read by then, and the waves must not part over it.
    if (found && wave == 0) {
      // the cheapest of the paths to the group in question, and how far behind the next one is
      const uint32_t target = p == 0 ? ov : uint32_t(sm.st[kSteps / 2 + p]) >> 4;
      u64 best = ~0ull, second = ~0ull;
      for (uint32_t i = lane; i < found; i += 64) {
        const u64 path = lists[(p & 1 ? kCloseList : 0) + i], key = (path & 0xffffffff00000000ull) | i;
        if ((uint32_t(path) & 0xfffu) != target) continue;
        second = min(second, max(best, key));
        best = min(best, key);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const u64 ob = __shfl_xor(best, o, 64), os = __shfl_xor(second, o, 64);
        second = min(min(second, os), max(best, ob));
        best = min(best, ob);
      }
      const uint32_t c = uint32_t(best >> 32), c2 = uint32_t(second >> 32);
      const uint32_t sum = p == 0 ? sat_add(start + 65536u, sat_add(c, margin)) : 0u;
      const bool good = __builtin_amdgcn_readfirstlane(int(sum <= limit && best != ~0ull && (second == ~0ull || c2 - c >= margin))) != 0;
      if (lane == 0) sm.close_ok = good;
      if (good) {
        // steps 0 .. p - 1 as the free path has them, then from path to path continued
        const uint16_t v = sm.st[kSteps / 2 + lane];
        if (int(lane) < p) sm.st[lane] = v;
        const uint32_t begin_lo = list0[lane], begin_hi = list0[lane + 64];
        uint32_t at = total + uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(best))));
        uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(paths[at])));
#pragma nounroll
        for (int q = p; q < kSteps; ++q) {
          const uint32_t g = lo & 0xfffu, k = (lo >> 12) & 0xffu;
          const uint32_t begin = uint32_t(__builtin_amdgcn_readlane(int(q + 1 < 64 ? begin_lo : begin_hi), (q + 1) & 63));
          at = q == kSteps - 1 ? 0u : begin + k;
          lo = q == kSteps - 1 ? ov : uint32_t(__builtin_amdgcn_readfirstlane(int(paths[at])));
          if (lane == 0) sm.st[q] = uint16_t((g << 4) | (lo & 15u));
        }
      }
    }
    __syncthreads();
    if (found) ok = __builtin_amdgcn_readfirstlane(int(sm.close_ok)) != 0;
  }
  return ok;
}
