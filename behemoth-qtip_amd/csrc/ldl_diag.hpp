// One workgroup's factorization of a diagonal block of the LDL on the device.  In a header of its own so that
// tests/cpp/diag_block_emulation.cpp can run it on the CPU, its waves in any order between two barriers.
#pragma once
#include <cstdint>

namespace qtipmi {
namespace {

// ---- the diagonal block: lower Cholesky of the kb x kb block at A (row stride ld; kb a multiple of 16, at most 256)
// and the inverses of its 16 x 16 diagonal blocks.  One workgroup: sub-panels of 16 columns, each factored by rows (a
// thread per row; every wave also carries the sub-panel's own 16 rows in its lanes' second set of registers, so that a
// column's values reach all lanes as scalars by lane reads, without a barrier between the columns), then subtracted
// from what lies right of it in 32 x 32 pieces, a wave each.
// Which products are rounded before the subtraction is the host's rule: for column j of the block and term p, with
// full = j & ~3: p < full always; of the j & 3 terms after that none for the diagonal element, and below it the first
// two if there are two or three.  full is a multiple of 4 and a sub-panel starts at a multiple of 16, so the terms of
// earlier sub-panels are always rounded and the rule only shows inside a sub-panel.
// Bound by its chain: 256 times a square root, a division and the update of the next column, 16 times a round trip of
// the sub-panel through memory.
constexpr int kDiag = 256, kSub = 16;

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u)), lane));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u >> 32)), lane));
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

using DiagLds = double[kSub][kDiag];  // [column of the sub-panel][row of the block], 32 KB
__device__ __forceinline__ void factor_diag_block(DiagLds& P, double* __restrict__ A, long ld, int kb,
                                                  double* __restrict__ rdiag, double* __restrict__ inv,
                                                  int* __restrict__ bad) {
  const int t = threadIdx.x, lane = t & 63, l16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  bool ok = true;
  for (int c0 = 0; c0 < kb; c0 += kSub) {
    double b[kSub];
    {
      const int r = c0 + t;
      const bool live = r < kb;
      double a[kSub];
      const double2* pa = reinterpret_cast<const double2*>(A + long(live ? r : c0) * ld + c0);
      const double2* pb = reinterpret_cast<const double2*>(A + long(c0 + l16) * ld + c0);
#pragma unroll
      for (int q = 0; q < kSub / 2; ++q) {
        const double2 va = pa[q], vb = pb[q];
        a[2 * q] = va.x, a[2 * q + 1] = va.y;
        b[2 * q] = vb.x, b[2 * q + 1] = vb.y;
      }
#pragma unroll
      for (int j = 0; j < kSub; ++j) {
        __builtin_amdgcn_sched_barrier(0);  // a column at a time: its lane values fill the scalar registers
        // the lane number anew: compared once for the whole loop, its sixteen masks would crowd those values out
        int me = l16;
        asm volatile("" : "+v"(me));
        const double d = lane_value(b[j], j);
        ok = ok && d > 0 && d <= 1.7976931348623157e308;
        const double l = __builtin_sqrt(d);
        a[j] = a[j] / l;
        // (the rows below only matter where they are stored, and the compiler would move all their arithmetic there,
        // with every lane value of all columns kept until then)
        asm volatile("" : "+v"(a[j]));
        b[j] = me == j ? l : b[j] / l;
#pragma unroll
        for (int jj = j + 1; jj < kSub; ++jj) {
          const double m = lane_value(b[j], jj);
          const int full = jj & ~3, rem = jj & 3;
          const bool rounded = j < full || j - full < (rem >= 2 ? 2 : 0);
          if (rounded) {
            a[jj] = a[jj] - m * a[j];
            const double below = b[jj] - m * b[j];
            b[jj] = j < full ? below : (me == jj ? __builtin_fma(-m, b[j], b[jj]) : below);
          } else {
            a[jj] = __builtin_fma(-m, a[j], a[jj]);
            b[jj] = __builtin_fma(-m, b[j], b[jj]);
          }
        }
      }
      if (t >= kSub && live) {
        double* out = A + long(r) * ld + c0;
#pragma unroll
        for (int q = 0; q < kSub / 2; ++q) reinterpret_cast<double2*>(out)[q] = make_double2(a[2 * q], a[2 * q + 1]);
#pragma unroll
        for (int j = 0; j < kSub; ++j) P[j][r] = a[j];
      }
    }
    __syncthreads();
    // the sub-panel's own rows are every wave's operand (pb), so they are replaced once all waves have them
    if (t < kSub) {
      double* out = A + long(c0 + t) * ld + c0;
      int me = t;
      asm volatile("" : "+v"(me));
#pragma unroll
      for (int j = 0; j < kSub; ++j)
        if (j <= me) out[j] = b[j];
    }
    // the part right of the sub-panel: rows and columns s0 .. kb - 1, lower triangle, tiles of 32 x 32 in a row-major
    // walk of the triangle, every fourth one this wave's; a lane owns 4 x 4 values
    const int s0 = c0 + kSub, T = (kb - s0 + 31) / 32, tiles = T * (T + 1) / 2;
    double c[2][4][4];
    auto place = [&](int idx, int& r, int& q) {
      int ti = 0;
      while ((ti + 1) * (ti + 2) / 2 <= idx) ++ti;
      r = s0 + 32 * ti + 4 * (lane >> 3);
      q = s0 + 32 * (idx - ti * (ti + 1) / 2) + 4 * (lane & 7);
    };
    auto fetch = [&](int idx, double (&v)[4][4]) {
      int r, q;
      place(idx, r, q);
      if (r < kb && q < kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double2* p = reinterpret_cast<const double2*>(A + long(r + i) * ld + q);
          const double2 x = p[0], y = p[1];
          v[i][0] = x.x, v[i][1] = x.y, v[i][2] = y.x, v[i][3] = y.y;
        }
      }
    };
    auto work = [&](int idx, double (&v)[4][4]) {
      int r, q;
      place(idx, r, q);
      if (r < kb && q < kb) {  // s0 and kb are multiples of 16: a lane's 4 x 4 values exist together or not at all
#pragma unroll
        for (int p = 0; p < kSub; ++p) {
          double x[4], y[4];
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            const double2 u = *reinterpret_cast<const double2*>(&P[p][r + i]);
            const double2 w = *reinterpret_cast<const double2*>(&P[p][q + i]);
            x[i] = u.x, x[i + 1] = u.y;
            y[i] = w.x, y[i + 1] = w.y;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = v[i][j] - x[i] * y[j];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          double2* p = reinterpret_cast<double2*>(A + long(r + i) * ld + q);
          p[0] = make_double2(v[i][0], v[i][1]);
          p[1] = make_double2(v[i][2], v[i][3]);
        }
      }
    };
    if (wave < tiles) fetch(wave, c[0]);
    for (int idx = wave; idx < tiles; idx += 8) {
      if (idx + 4 < tiles) fetch(idx + 4, c[1]);
      work(idx, c[0]);
      if (idx + 4 < tiles) {
        if (idx + 8 < tiles) fetch(idx + 8, c[0]);
        work(idx + 4, c[1]);
      }
    }
    __syncthreads();  // (orders the stores above before the next sub-panel's loads as well: one compute unit)
  }
  if (!ok && lane == 0) *bad = 1;
  if (t < kb) rdiag[t] = 1.0 / A[long(t) * ld + t];
  // column t % 16 of the inverse of diagonal block t / 16, by forward substitution; every sum one fused chain
  if (t < kb) {
    const int b0 = t & ~15, cc = t & 15;
    double V[kSub];
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      const double* row = A + long(b0 + i) * ld + b0;
      double s = i == cc ? 1.0 : 0.0;
#pragma unroll
      for (int p = 0; p < i; ++p) s = __builtin_fma(-row[p], V[p], s);
      V[i] = s / row[i];
      inv[long(b0 + i) * 16 + cc] = V[i];
    }
  }
}

}  // namespace
}  // namespace qtipmi
