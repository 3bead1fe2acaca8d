// The fp64 block LDL of the group quantizer and the Cholesky factorization of the NVFP4 calibration on the device, in
// the order of operations of the host factorization (host_ldl.cpp, host_ldl_diag.cpp; reference
// src/qtip_core.cpp:321-487): the factor is the host's bit for bit.  Right-looking panels of 256 columns, three
// launches per panel on one stream (two where the trailing matrix is large: its update brings the next diagonal block with
// it) and nothing that goes through the host:
//   ldl_diag_kernel          the 256 x 256 diagonal block (one workgroup)
//   ldl_solve_kernel         the rows below it, and the panel's columns of L
//   rank_update_lower_kernel the trailing matrix
// v_mfma_f64_16x16x4_f64 accumulates its four products like a chain of fused multiply-adds in ascending k (checked bit
// for bit against std::fma chains), which is how the host's micro-kernels form every element of an update and its
// panel solve every partial sum; where the host rounds a product before it subtracts it (the diagonal block) the
// vector units do the same.  Division and square root are correctly rounded on both.
//
// The form it replaced kept the panels on the host (3.3 GB of panel columns down and up per factorization at n = 28672,
// the diagonal blocks on one core) and only updated here.  n = 1024 / 4096 / 12288 / 28672, rotated Hessian on the
// device, L on the device and in page-locked host memory: 1.5 / 5.8 / 26.2 / 161 ms against 2.9 / 16.4 / 81 / 361 ms.
// The copy of L down, which the group calls do not ask for, runs beside it.  A panel's diagonal block
// takes 0.20 ms, its solve 0.08 ms (4096 rows), its update runs at 57 TFLOP/s of the card's 71 (a large fp64 product).
#include <algorithm>
#include <utility>
#include <vector>

#include "quantizer_impl.hpp"
#include "ldl_diag.hpp"

namespace qtipmi {
namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));

// A[i][j] = (H[i][j] + H[j][i]) / 2 in fp64, lower triangle (symmetrize_lower_host); the factorization's flag is cleared
__global__ void symmetrize_lower_kernel(const float* __restrict__ H, long n, double* __restrict__ A, int* __restrict__ bad) {
  const long j = long(blockIdx.x) * blockDim.x + threadIdx.x, i = blockIdx.y;
  if (i == 0 && j == 0) *bad = 0;
  if (j > i || j >= n) return;
  A[i * n + j] = 0.5 * (double(H[i * n + j]) + double(H[j * n + i]));
}

// C -= acc for a wave's 64 x 64 outputs (rows i0 .., columns j0 ..; only i < nr, j <= i exist).  A block that lies
// inside the triangle altogether (nearly all do) fetches the 16 values of a row block together, so it waits for 4
// round trips to memory, not 64; the others go element by element.
__device__ __forceinline__ void subtract_tile(const double4_t (&acc)[4][4], double* __restrict__ C, long ldc, int nr,
                                              int i0, int j0, int lane) {
  if (i0 + 64 <= nr && j0 + 63 <= i0) {  // the same for the whole wave
    double* base = C + long(i0 + (lane >> 4)) * ldc + j0 + (lane & 15);
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      double c[4][4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double* row = base + long(mi * 16 + 4 * v) * ldc;
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) c[ni][v] = row[ni * 16];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double* row = base + long(mi * 16 + 4 * v) * ldc;
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) row[ni * 16] = c[ni][v] - acc[mi][ni][v];
      }
    }
    return;
  }
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gi = i0 + mi * 16 + (lane >> 4) + 4 * v, gj = j0 + ni * 16 + (lane & 15);
        if (gi < nr && gj <= gi) C[long(gi) * ldc + gj] -= acc[mi][ni][v];
      }
}

// C[i][j] -= sum_p X[i][p] * X[j][p] for one 128 x 128 tile of the nr x nr lower triangle, every element one chain
// over p = 0 .. kb-1 from zero, then one subtraction.  Xt: kb x nr (the transposed solved rows, row stride ldx; nr and
// ldx multiples of 4, kb a multiple of 8), C: row stride ldc.  The grid enumerates the tiles
// (bi, bj <= bi) of the triangle.
// 256 threads, 2 x 2 waves of 64 x 64.  The workgroups share the chip with the Viterbi kernel's (168 registers, 50 KB
// of LDS each, three per CU), so this one stays within 168 registers and 48 KB of LDS and takes the place of one of
// them, not two: the operand slices go from global memory straight into LDS (global_load_lds_dwordx4: a wave's 64
// lanes fill one 1 KB row of 128 doubles), eight columns of the panel per stage, three stages in flight, one
// barrier per stage, no staging registers; fragment reads and loads go one at a time under the MFMAs (see the loop).
// Lanes beyond nr in the last tile row read whatever follows in Xt (the caller's buffer extends at least 128 doubles
// beyond the last row read); those columns only feed outputs that are never stored.
constexpr int UT = 128;
constexpr int VK = 8, VSTAGES = 3;
using UpdateLds = double[VSTAGES][2][VK][UT];  // [stage][Xi | Xj][k][column], 48 KB
__device__ __forceinline__ void update_tile(UpdateLds& S, const double* __restrict__ Xt, long ldx, int nr, int kb,
                                            double* __restrict__ C, long ldc, int bi, int bj) {
  const int i0 = bi * UT, j0 = bj * UT;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 1, wn = wave & 1;
  double4_t acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = double4_t{0, 0, 0, 0};
  // wave w brings rows 2w and 2w + 1 of a stage's Xi and Xj slices; gi / gj: this lane's piece of the next slice to
  // be requested, `asked` its number
  const double* gi = Xt + long(2 * wave) * ldx + i0 + 2 * lane;
  const double* gj = Xt + long(2 * wave) * ldx + j0 + 2 * lane;
  const long slice_stride = long(VK) * ldx;
  int asked = 0;
  typedef __attribute__((address_space(3))) void* lds_ptr;
  auto load1 = [&](int st, int q) {  // into stage st; q = 0, 1: rows 2w, 2w + 1 of Xi; 2, 3: of Xj
    const int r = q & 1;
    if (q < 2) __builtin_amdgcn_global_load_lds(gi + r * ldx, (lds_ptr)&S[st][0][2 * wave + r][0], 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(gj + r * ldx, (lds_ptr)&S[st][1][2 * wave + r][0], 16, 0, 0);
  };
  auto asked_one = [&] {
    gi += slice_stride, gj += slice_stride, ++asked;
    // the two running pointers as they are: without this the compiler keeps one pointer per load of the unrolled
    // loop, two dozen registers that the accumulators leave no room for
    asm volatile("" : "+v"(gi), "+v"(gj));
  };
  const int slices = kb / VK;  // kb is a multiple of 16
  // fragments of the 4 k of step ks (0, 1) of the slice in stage st: a[set][mi], b[set][ni]
  const int c16 = lane & 15, kq = lane >> 4;
  double fa[2][4], fb[2][4];
  auto read1 = [&](int st, int ks, int set, int j) {  // j = 0..7 in the order the MFMAs first use them: a0 b0 b1 b2 b3 a1 a2 a3
    const int kr = 4 * ks + kq;
    if (j == 0 || j >= 5) {
      const int mi = j == 0 ? 0 : j - 4;
      fa[set][mi] = S[st][0][kr][wm * 64 + mi * 16 + c16];
    } else {
      const int ni = j - 1;
      fb[set][ni] = S[st][1][kr][wn * 64 + ni * 16 + c16];
    }
  };
  auto mfma = [&](int set, int j) {
    const int mi = j >> 2, ni = j & 3;
    acc[mi][ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[set][mi], fb[set][ni], acc[mi][ni], 0, 0, 0);
  };
  // Slices 0 and 1 requested, slice 0 landed (this wave's loads, then everyone's: a bare barrier, which does not wait
  // for the loads still in flight), slice 2 requested, the fragments of slice 0's first 4 k read.
  load1(0, 0), load1(0, 1), load1(0, 2), load1(0, 3);
  asked_one();
  if (slices > 1) {
    load1(1, 0), load1(1, 1), load1(1, 2), load1(1, 3);
    asked_one();
  }
  if (slices > 1) __builtin_amdgcn_s_waitcnt(0x0F74);  // vmcnt(4)
  else __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (asked < slices) {
    load1(2, 0), load1(2, 1), load1(2, 2), load1(2, 3);
    asked_one();
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) read1(0, 0, 0, j);
  // One slice: 32 MFMAs, two steps of 4 k on fragment sets 0 and 1.  The workgroup runs beside the Viterbi kernel's,
  // one wave per SIMD with nothing to hide a wait behind but its own MFMAs (32 cycles each, during which the wave may
  // issue other work): under every other MFMA of a step it reads one fragment of the next step, and under MFMAs 1, 5,
  // 9, 13 of the second step it requests one row of slice sl + 3 - after the barrier in the middle, which says slice
  // sl + 1 has landed everywhere and every wave has asked for its last fragments of slice sl, whose stage is
  // therefore free.  The scheduling barriers pin that order.  kSteady: every slice asked for exists and one more is
  // on its way beyond sl + 1, so vmcnt(4) = "slice sl + 1 is here"; the last slices run the same code with the
  // conditions and a full wait.
#define QTIP_SB __builtin_amdgcn_sched_barrier(0)
  auto slice = [&](auto steady, auto stage, int sl) {  // slice sl, which lies in stage sl % VSTAGES = stage
    constexpr bool kSteady = decltype(steady)::value;
    constexpr int st = decltype(stage)::value, nst = (st + 1) % VSTAGES;
    const bool next = kSteady || sl + 1 < slices;
#define QTIP_M0(j) { mfma(0, j); QTIP_SB; }
#define QTIP_R0(j) { mfma(0, j); QTIP_SB; read1(st, 1, 1, (j) / 2); QTIP_SB; }
    QTIP_SB;
    QTIP_R0(0) QTIP_M0(1) QTIP_R0(2) QTIP_M0(3) QTIP_R0(4) QTIP_M0(5) QTIP_R0(6) QTIP_M0(7)
    QTIP_R0(8) QTIP_M0(9) QTIP_R0(10) QTIP_M0(11) QTIP_R0(12) QTIP_M0(13) QTIP_R0(14) QTIP_M0(15)
    if (next) {
      // this wave's part of slice sl + 1 has landed and its reads of slice sl have returned
      if (kSteady) __builtin_amdgcn_s_waitcnt(0x0074);  // vmcnt(4) lgkmcnt(0)
      else __builtin_amdgcn_s_waitcnt(0x0070);          // vmcnt(0) lgkmcnt(0)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    const bool go = kSteady || asked < slices;
#define QTIP_M1(j) { mfma(1, j); QTIP_SB; }
#define QTIP_R1(j) { mfma(1, j); QTIP_SB; if (next) read1(nst, 0, 0, (j) / 2); QTIP_SB; }
#define QTIP_L1(j) { mfma(1, j); QTIP_SB; if (go) load1(st, ((j) - 1) / 4); QTIP_SB; }
    QTIP_SB;
    QTIP_R1(0) QTIP_L1(1) QTIP_R1(2) QTIP_M1(3) QTIP_R1(4) QTIP_L1(5) QTIP_R1(6) QTIP_M1(7)
    QTIP_R1(8) QTIP_L1(9) QTIP_R1(10) QTIP_M1(11) QTIP_R1(12) QTIP_L1(13) QTIP_R1(14) QTIP_M1(15)
    if (go) asked_one();
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  static_assert(VSTAGES == 3);
  int sl = 0;
  for (; sl + 5 < slices; sl += 3) {
    slice(std::true_type{}, S0{}, sl);
    slice(std::true_type{}, S1{}, sl + 1);
    slice(std::true_type{}, S2{}, sl + 2);
  }
  for (; sl < slices; sl += 3) {  // the last 3 to 5 slices (or all, of fewer)
    slice(std::false_type{}, S0{}, sl);
    if (sl + 1 < slices) slice(std::false_type{}, S1{}, sl + 1);
    if (sl + 2 < slices) slice(std::false_type{}, S2{}, sl + 2);
  }
#undef QTIP_M0
#undef QTIP_R0
#undef QTIP_M1
#undef QTIP_R1
#undef QTIP_L1
#undef QTIP_SB
  // the lane number anew: the loop leaves no register to keep it in
  const int ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  subtract_tile(acc, C, ldc, nr, i0 + wm * 64, j0 + wn * 64, ln);
}

__global__ __launch_bounds__(256, 3) void ldl_diag_kernel(double* __restrict__ A, long ld, int kb,
                                                          double* __restrict__ rdiag, double* __restrict__ inv,
                                                          int* __restrict__ bad) {
  __shared__ __attribute__((aligned(16))) DiagLds P;
  factor_diag_block(P, A, ld, kb, rdiag, inv, bad);
}

__device__ __forceinline__ void triangle_tile(int tile, int& bi, int& bj) {
  // row bi with bi (bi + 1) / 2 <= tile: the square root in fp32, then one step either way
  bi = int((__builtin_sqrtf(8.0f * float(tile) + 1.0f) - 1.0f) * 0.5f);
  while (bi * (bi + 1) / 2 > tile) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= tile) ++bi;
  bj = tile - bi * (bi + 1) / 2;
}
__global__ __launch_bounds__(256, 3) void rank_update_lower_kernel(const double* __restrict__ Xt, long ldx, int nr,
                                                                     int kb, double* __restrict__ C, long ldc) {
  __shared__ __attribute__((aligned(16))) UpdateLds S;
  int bi, bj;
  triangle_tile(blockIdx.x, bi, bj);
  update_tile(S, Xt, ldx, nr, kb, C, ldc, bi, bj);
}
// The update of a large trailing matrix with the next panel's diagonal block: the first workgroup updates the three tiles
// of the leading 256 x 256 block and factors it while the others update the rest.  Two launches a panel instead of three
// with the diagonal block's 0.2 ms under the update - and, beside the quantization of another group, whose Viterbi
// workgroups fill the chip, a launch waits some milliseconds for their places, so the launches are what the factorization
// takes there (12288 x 28672 groups in a row: 1.34 -> 1.28 s a factorization; alone at n = 28672 169 -> 156 ms).
__global__ __launch_bounds__(256, 3) void rank_update_next_diag_kernel(const double* __restrict__ Xt, long ldx, int nr,
                                                                       int kb, double* __restrict__ C, long ldc,
                                                                       double* __restrict__ rdiag, double* __restrict__ inv,
                                                                       int* __restrict__ bad) {
  __shared__ __attribute__((aligned(16))) UpdateLds S;
  if (blockIdx.x == 0) {
#pragma nounroll
    for (int tile = 0; tile < 3; ++tile) {
      update_tile(S, Xt, ldx, nr, kb, C, ldc, tile > 0, tile > 1);
      __syncthreads();  // the next tile's operands take the place of this one's, and the block is whole after the last
    }
    static_assert(sizeof(DiagLds) <= sizeof(UpdateLds) && kDiag == 2 * UT);
    factor_diag_block(*reinterpret_cast<DiagLds*>(&S), C, ldc, kDiag, rdiag, inv, bad);
  } else {
    int bi, bj;
    triangle_tile(blockIdx.x + 2, bi, bj);
    update_tile(S, Xt, ldx, nr, kb, C, ldc, bi, bj);
  }
}

// ---- the rows below the diagonal block: X L11^T = A21, every element x_j = ((s0 + s1) + (s2 + s3)) / l_jj (times the
// reciprocal), s_(p mod 4) a chain of fused multiply-adds over the full groups of four p < j, the p left over added to
// s0's: the four sums of the 16 columns of a block over all earlier blocks are four chains on the matrix cores (k = the
// four p of a block that share p mod 4), and only the 16 x 16 triangle of the block itself runs on the vector units.
// One wave takes 16 rows; its solved values stay in LDS as the next blocks' operand (45.6 KB in all: three waves per
// compute unit, or one in the place of a Viterbi workgroup).  It leaves them transposed for the update kernel (Xt, row
// stride ldx) and forms the panel's columns of the result from them:
//   kScalar false: L = C blockdiag(C_bb^-1), a chain of 16 fused multiply-adds per value (again the matrix cores)
//   kScalar true:  L_ij = C_ij / C_jj, and dw_j = C_jj^2
// The first kb / 16 workgroups take the rows of the diagonal block itself, which are solved already.  A, L, dw: at the
// panel's diagonal; L comes zeroed.
// Bound by the chain of a wave: 16 triangles of 16 dependent columns and 480 dependent matrix instructions.
constexpr int kXStride = 17;  // doubles per solved column in LDS: 16 rows and one of padding
template <bool kScalar>
__global__ __launch_bounds__(64) void ldl_solve_kernel(const double* __restrict__ A, long ld, int kb,
                                                       const double* __restrict__ rdiag, const double* __restrict__ inv,
                                                       double* __restrict__ Xt, long ldx, float* __restrict__ L, long ldl,
                                                       float* __restrict__ dw, int* __restrict__ bad) {
  __shared__ double X[kDiag * kXStride];  // X[p * kXStride + row]
  __shared__ double S[4][kSub][kXStride];  // the four partial sums of a block's columns [chain][column][row]
  __shared__ __attribute__((aligned(16))) double D[kSub][kSub];  // the block's own triangle of L11
  const int lane = threadIdx.x, q = lane >> 4, r = lane & 15;
  const int nd = kb / 16, blocks = nd;
  const bool below = int(blockIdx.x) >= nd;
  const int row0 = 16 * int(blockIdx.x);  // relative to the panel's diagonal
  const double* rows = A + long(row0) * ld;
  int last = blocks;  // blocks of this wave's rows that hold values of C strictly left of their own diagonal block
  if (below) {
    double init[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) init[v] = rows[long(r) * ld + q + 4 * v];
    double2 tri[2] = {*reinterpret_cast<const double2*>(A + long(r) * ld + 4 * q),
                      *reinterpret_cast<const double2*>(A + long(r) * ld + 4 * q + 2)};
    // row j0 + r of L11, the four p of block pb that start at 4 q: one 32-byte piece, fetched kDepth blocks ahead; the
    // first kDepth of a block of columns are fetched before the triangle of the block before it
    constexpr int kDepth = 4;
    double2 f[kDepth][2];
#pragma unroll
    for (int i = 0; i < kDepth; ++i) f[i][0] = f[i][1] = make_double2(0.0, 0.0);
    for (int jb = 0; jb < blocks; ++jb) {
      const int j0 = 16 * jb;
      double4_t s[4];
      s[0] = double4_t{init[0], init[1], init[2], init[3]};
#pragma unroll
      for (int c = 1; c < 4; ++c) s[c] = double4_t{0, 0, 0, 0};
      if (jb + 1 < blocks) {
#pragma unroll
        for (int v = 0; v < 4; ++v) init[v] = rows[long(r) * ld + j0 + 16 + q + 4 * v];
      }
      *reinterpret_cast<double2*>(&D[r][4 * q]) = tri[0];
      *reinterpret_cast<double2*>(&D[r][4 * q + 2]) = tri[1];
      if (jb + 1 < blocks) {
        const double* next = A + long(j0 + 16 + r) * ld + j0 + 16 + 4 * q;
        tri[0] = *reinterpret_cast<const double2*>(next);
        tri[1] = *reinterpret_cast<const double2*>(next + 2);
      }
      const double rd = rdiag[j0 + r];
      const double* lrow = A + long(j0 + r) * ld + 4 * q;
      for (int pb0 = 0; pb0 < jb; pb0 += kDepth) {
#pragma unroll
        for (int i = 0; i < kDepth; ++i) {
          const int pb = pb0 + i;
          if (pb < jb) {
            const double2 u = f[i][0], w = f[i][1];
            if (pb + kDepth < jb) {
              f[i][0] = *reinterpret_cast<const double2*>(lrow + 16 * (pb + kDepth));
              f[i][1] = *reinterpret_cast<const double2*>(lrow + 16 * (pb + kDepth) + 2);
            }
            const double* x = X + (16 * pb + 4 * q) * kXStride + r;
            s[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.x, x[0], s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.y, x[kXStride], s[1], 0, 0, 0);
            s[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(-w.x, x[2 * kXStride], s[2], 0, 0, 0);
            s[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(-w.y, x[3 * kXStride], s[3], 0, 0, 0);
          }
        }
      }
      // a lane holds columns q + 4 v of row r: through LDS, so that every lane has all 16 columns of its row (the four
      // quarters of the wave then do the same)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) S[c][q + 4 * v][r] = s[c][v];
      if (jb + 1 < blocks) {
        const double* next = A + long(j0 + 16 + r) * ld + 4 * q;
#pragma unroll
        for (int i = 0; i < kDepth; ++i)
          if (i < jb + 1) {
            f[i][0] = *reinterpret_cast<const double2*>(next + 16 * i);
            f[i][1] = *reinterpret_cast<const double2*>(next + 16 * i + 2);
          }
      }
      __syncthreads();
      // the partial sums and the row of the triangle of column j + 1 are read from LDS while column j is worked on (the
      // empty asm keeps it at that: all rows at once do not fit the registers)
      double x[kSub], lj[2][kSub], part[2][4];
#pragma unroll
      for (int c = 0; c < 4; ++c) part[0][c] = S[c][0][r];
#pragma unroll
      for (int j = 0; j < kSub; ++j) {
        const int cur = j & 1, nxt = cur ^ 1;
        if (j + 1 < kSub) {
#pragma unroll
          for (int c = 0; c < 4; ++c) part[nxt][c] = S[c][j + 1][r];
#pragma unroll
          for (int p = 0; p <= j; ++p) lj[nxt][p] = D[j + 1][p];
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        double(&s4)[4] = part[cur];
#pragma unroll
        for (int p = 0; p < (j & ~3); ++p) s4[p & 3] = __builtin_fma(-lj[cur][p], x[p], s4[p & 3]);
#pragma unroll
        for (int p = j & ~3; p < j; ++p) s4[0] = __builtin_fma(-lj[cur][p], x[p], s4[0]);
        x[j] = ((s4[0] + s4[1]) + (s4[2] + s4[3])) * lane_value(rd, j);
      }
#pragma unroll
      for (int j = 0; j < kSub; ++j)
        if (q == (j & 3)) X[(j0 + j) * kXStride + r] = x[j];
      __syncthreads();
    }
    double* xt = Xt + (row0 - kb) + r;
    for (int p = q; p < kb; p += 4) xt[long(p) * ldx] = X[p * kXStride + r];
  } else {
    // the finished rows of the diagonal block (with their own block, of which the scalar form takes the lower part)
    last = int(blockIdx.x);
    const int cols = 16 * (last + 1);
    for (int i = 0; i < 16; ++i)
      for (int p = lane; p < cols; p += 64) X[p * kXStride + i] = rows[long(i) * ld + p];
    __syncthreads();
  }
  if constexpr (kScalar) {
    for (int i = 0; i < 16; ++i) {
      const int end = below ? kb : row0 + i;
      float* out = L + long(row0 + i) * ldl;
      for (int p = lane; p < end; p += 64) out[p] = float(X[p * kXStride + i] / A[long(p) * ld + p]);
    }
    if (!below && lane < 16) {
      const double d = X[(row0 + lane) * kXStride + lane];
      dw[row0 + lane] = float(d * d);
    }
  } else {
    bool finite = true;
    for (int b = 0; b < last; ++b) {
      double4_t o = double4_t{0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int p = 4 * m + q;
        o = __builtin_amdgcn_mfma_f64_16x16x4f64(X[(16 * b + p) * kXStride + r], inv[long(16 * b + p) * 16 + r], o, 0, 0,
                                                 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        L[long(row0 + q + 4 * v) * ldl + 16 * b + r] = float(o[v]);
        finite = finite && o[v] * 0.0 == 0.0;
      }
    }
    if (!finite) *bad = 1;
  }
}

__global__ void add_to_diagonal_kernel(double* __restrict__ A, long n, double v) {
  const long i = blockIdx.x * long(blockDim.x) + threadIdx.x;
  if (i < n) A[i * n + i] += v;
}

}  // namespace

namespace {
// Factors the symmetric matrix whose lower triangle lies in c->ldl_A (n x n) on stream s, *c->ldl_bad cleared.  L (n x n fp32, device)
// receives the block LDL's factor, or with dw the scalar one's; everything outside its strict (block) lower triangle is
// zero.  host_L (optional) receives L as well: the rows of a panel's diagonal block are final once the panel is solved, and
// go down from a stream of their own, 1024 at a time, while the factorization runs on (n = 28672 into pageable memory:
// host buffers in and out 0.59 -> 0.44 s, page-locked L alone 216 -> 161 ms; up to n = 1024 there is one such block, and it
// follows on s).  Waits for the stream; false if the matrix is not positive definite.
bool factor_on_device(qtip_ctx* c, long n, float* L, float* dw, hipStream_t s, float* host_L = nullptr) {
  struct RowsDown {  // whatever ends the call, nothing of it is left behind
    hipStream_t stream = nullptr;
    std::vector<std::pair<long, hipEvent_t>> ready;  // (rows final, after this event)
    ~RowsDown() {
      if (stream) (void)hipStreamSynchronize(stream);
      for (auto& r : ready) (void)hipEventDestroy(r.second);
    }
  } down;
  constexpr long kRowsDown = 1024;
  if (host_L && n > kRowsDown) {
    if (!c->ldl_down_stream) QTIP_HIP(hipStreamCreateWithFlags(&c->ldl_down_stream, hipStreamNonBlocking));
    down.stream = c->ldl_down_stream;
  }
  QTIP_HIP(hipMemsetAsync(L, 0, size_t(n) * n * sizeof(float), s));
  bool diag_done = false;  // this panel's diagonal block came with the update before it
  int turn = 0;            // the reciprocals and inverses of a panel and of the one factored beside its update
  for (long k = 0; k < n; k += kDiag, turn ^= 1) {
    const int kb = int(std::min<long>(kDiag, n - k));
    const long nr = n - k - kb;
    double* const D = c->ldl_A.p + k * n + k;
    const size_t set = size_t(kDiag) * 17;
    double *const rdiag = c->ldl_diag.p + turn * set, *const inv = rdiag + kDiag;
    if (!diag_done) {
      ldl_diag_kernel<<<dim3(1), dim3(256), 0, s>>>(D, n, kb, rdiag, inv, c->ldl_bad.p);
      QTIP_HIP(hipGetLastError());
    }
    const dim3 grid(unsigned((kb + nr) / 16));
    const auto solve = dw ? ldl_solve_kernel<true> : ldl_solve_kernel<false>;
    solve<<<grid, dim3(64), 0, s>>>(D, n, kb, rdiag, inv, c->ldl_Xt.p, nr, L + k * n + k, n, dw ? dw + k : nullptr,
                                    c->ldl_bad.p);
    QTIP_HIP(hipGetLastError());
    if (down.stream && (nr <= 0 || (k + kb) % kRowsDown == 0)) {
      hipEvent_t e;
      QTIP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      down.ready.emplace_back(k + kb, e);
      QTIP_HIP(hipEventRecord(e, s));
    }
    if (nr <= 0) break;
    const long nt = (nr + UT - 1) / UT;
    // what the update kernel assumes: whole stages of 8 panel columns, 16-byte aligned rows of Xt, and readable memory
    // up to the end of the last tile row's 128 columns in every row of Xt
    QTIP_REQUIRE(kb % VK == 0 && nr % 4 == 0 && size_t(kb - 1) * nr + size_t(nt) * UT <= c->ldl_Xt.n,
                 "LDL update: operand shape the kernel does not cover (kb = %d, nr = %ld)", kb, nr);
    double* const C = c->ldl_A.p + (k + kb) * n + k + kb;
    // three tiles in a row and a diagonal block take one workgroup 0.28 ms, a diagonal block by itself 0.20 ms after the
    // update: even at about 6000 rows (1176 tiles, 0.1 ms), all of the 0.2 ms hidden from 12000 rows on
    diag_done = nr >= 6144;
    if (diag_done) {
      double* const next = c->ldl_diag.p + (turn ^ 1) * set;
      rank_update_next_diag_kernel<<<dim3(unsigned(nt * (nt + 1) / 2 - 2)), dim3(256), 0, s>>>(
          c->ldl_Xt.p, nr, int(nr), kb, C, n, next, next + kDiag, c->ldl_bad.p);
    } else {
      rank_update_lower_kernel<<<dim3(unsigned(nt * (nt + 1) / 2)), dim3(256), 0, s>>>(c->ldl_Xt.p, nr, int(nr), kb, C, n);
    }
    QTIP_HIP(hipGetLastError());
  }
  long row = 0;
  for (const auto& r : down.ready) {
    QTIP_HIP(hipEventSynchronize(r.second));
    QTIP_HIP(hipMemcpyAsync(host_L + size_t(row) * n, L + size_t(row) * n, size_t(r.first - row) * n * sizeof(float),
                            hipMemcpyDeviceToHost, down.stream));
    row = r.first;
  }
  if (down.stream) QTIP_HIP(hipStreamSynchronize(down.stream));
  else if (host_L) QTIP_HIP(hipMemcpyAsync(host_L, L, size_t(n) * n * sizeof(float), hipMemcpyDeviceToHost, s));
  int bad = 0;
  QTIP_HIP(hipMemcpyAsync(&bad, c->ldl_bad.p, sizeof bad, hipMemcpyDeviceToHost, s));
  QTIP_HIP(hipStreamSynchronize(s));
  return bad == 0;
}

hipStream_t factor_stream(qtip_ctx* c, long n) {
  if (!c->ldl_stream) QTIP_HIP(hipStreamCreateWithFlags(&c->ldl_stream, hipStreamNonBlocking));
  c->ldl_A.ensure(size_t(n) * n);
  c->ldl_Xt.ensure(size_t(n) * kDiag);
  c->ldl_diag.ensure(2 * size_t(kDiag) * 17);
  c->ldl_bad.ensure(1);
  return c->ldl_stream;
}

// whatever ends the scope, nothing queued on the stream outlives the buffers of the call
struct Settle {
  hipStream_t s;
  ~Settle() { (void)hipStreamSynchronize(s); }
};
}  // namespace

void reserve_device_ldl(qtip_ctx* c, int n) { (void)factor_stream(c, n); }

// The Hessian preparation of the calibrated NVFP4 quantizer (nvfp4_prepare_host) on the device: the same chains, hence
// the same L and dw bit for bit.  dev_L (n x n), dev_dw: device buffers of the caller, or null for the context's own;
// host_L, host_dw: optional, or both with the context's own buffers.
void nvfp4_prepare_device_impl(qtip_ctx* c, const float* host_H, int n, double sigma_reg, float* dev_L, float* dev_dw,
                               float* host_L, float* host_dw) {
  QTIP_REQUIRE(c && host_H && ((dev_L && dev_dw) || (host_L && host_dw)) && n > 0 && n % 16 == 0,
               "nvfp4_prepare (device): bad arguments (n = %d)", n);
  QTIP_REQUIRE(n <= 65535, "nvfp4_prepare (device): n = %d is beyond one grid dimension", n);
  double dsum = 0;
  for (int i = 0; i < n; ++i) dsum += host_H[size_t(i) * n + i];
  const double creg = sigma_reg * dsum / n;
  hipStream_t s = factor_stream(c, n);
  Settle settle{s};
  const size_t nn = size_t(n) * n;
  if (!dev_L || !dev_dw) {
    c->ldl_L.ensure(nn + size_t(n));
    dev_L = c->ldl_L.p, dev_dw = dev_L + nn;
  }
  c->ldl_H.ensure(nn);
  QTIP_HIP(hipMemcpyAsync(c->ldl_H.p, host_H, size_t(n) * n * 4, hipMemcpyHostToDevice, s));
  symmetrize_lower_kernel<<<dim3(unsigned((n + 255) / 256), unsigned(n)), dim3(256), 0, s>>>(c->ldl_H.p, n, c->ldl_A.p,
                                                                                           c->ldl_bad.p);
  QTIP_HIP(hipGetLastError());
  add_to_diagonal_kernel<<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, s>>>(c->ldl_A.p, n, creg);
  QTIP_HIP(hipGetLastError());
  if (!factor_on_device(c, n, dev_L, dev_dw, s, host_L))
    throw Error(QTIP_E_NOT_PD, "NVFP4 calibration: Hessian not positive definite");
  if (host_dw) {
    QTIP_HIP(hipMemcpyAsync(host_dw, dev_dw, size_t(n) * 4, hipMemcpyDeviceToHost, s));
    QTIP_HIP(hipStreamSynchronize(s));
  }
}

// The block LDL of the rotated Hessian: dev_HRr, or host_HRr if that is null.  L goes to host_L, to dev_L (n x n device
// buffer), or to both.  (Without dev_L it is formed in a buffer the context keeps: one made and freed here would have the
// free wait for everything on the device, the quantization of another group included.)
void ldl_hessian_device_impl(qtip_ctx* c, const float* host_HRr, int n, float* host_L, const float* dev_HRr, float* dev_L) {
  QTIP_REQUIRE(c && n > 0 && n % 16 == 0 && (host_HRr || dev_HRr) && (host_L || dev_L),
               "ldl_hessian (device): bad arguments (n = %d)", n);
  QTIP_REQUIRE(n <= 65535, "ldl_hessian (device): n = %d is beyond one grid dimension", n);
  hipStream_t s = factor_stream(c, n);
  const size_t nn = size_t(n) * n;
  Settle settle{s};
  if (!dev_L) {
    c->ldl_L.ensure(nn);
    dev_L = c->ldl_L.p;
  }
  if (!dev_HRr) {
    c->ldl_H.ensure(nn);
    QTIP_HIP(hipMemcpyAsync(c->ldl_H.p, host_HRr, nn * 4, hipMemcpyHostToDevice, s));
  }
  symmetrize_lower_kernel<<<dim3(unsigned((n + 255) / 256), unsigned(n)), dim3(256), 0, s>>>(
      dev_HRr ? dev_HRr : c->ldl_H.p, n, c->ldl_A.p, c->ldl_bad.p);
  QTIP_HIP(hipGetLastError());
  if (!factor_on_device(c, n, dev_L, nullptr, s, host_L)) throw Error(QTIP_E_NOT_PD, "block LDL failed (H not PD)");
}

}  // namespace qtipmi
