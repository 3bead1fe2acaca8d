// NVFP4 fallback quantizer on the device: scale search and Hessian-calibrated rounding (reference:
// nvfp4_quantize_group, nv_block_kernel and nv_feedback_kernel, src/nvfp4_gpu.hip:66-243; format src/nvfp4.hpp).
// Every fp32 operation is the reference kernel's, in its order.  The reference builds with hipcc's default
// floating-point contraction, which turns its three "sum += a * b" statements (block feedback, cost, column
// feedback) into fused multiply-adds; this file is built without contraction and writes those three as fmaf, so
// the bytes equal both the reference's gfx950 build and a CPU evaluation of the same formulas.
//
// Layout: the reference walks row-major W with one thread per matrix row, so neighbouring lanes are n floats apart.
// Here W, the feedback F and the outputs live transposed on the device ([column][row]): a wave's 64 rows are one
// 256-byte line for every column it touches.  Columns are processed in 16-wide blocks from the last to the first;
// the residual of a finished block goes to all remaining columns before the next block starts.
#include <algorithm>

#include "misc.hpp"
#include "nvfp4_codec.hpp"
#include "qtip_internal.hpp"

namespace qtipmi {
namespace {

// The scalar codec is nvfp4_codec.hpp's: e4m3_value (code <= 126 -> value), e4m3_of_magnitude (finite x -> code of |x|),
// through_bf16, e2m1_value and e2m1_of_magnitude (a >= 0 -> code).
namespace nvc = nvcodec;

constexpr int kScaleTries = 11;  // scale candidates of the search: the plain one, 8 shrink factors, one code down, one up
constexpr int kBlockRows = 64;  // matrix rows per workgroup: one per lane

// Block scale candidate number `which` (uniform over a wave) of a row whose 16 targets have the largest magnitude
// amax; the list and its order are the reference's (src/nvfp4_gpu.hip:97-105).
__device__ __forceinline__ unsigned nv_candidate(int which, float amax, float global) {
  if (which >= 1 && which <= 8) {
    float shrink = 1.05f;
    switch (which) {
      case 1: shrink = 0.70f; break;
      case 2: shrink = 0.75f; break;
      case 3: shrink = 0.80f; break;
      case 4: shrink = 0.85f; break;
      case 5: shrink = 0.90f; break;
      case 6: shrink = 0.95f; break;
      case 7: shrink = 1.00f; break;
      default: break;
    }
    return nvc::e4m3_of_magnitude(amax * shrink / (6.f * global));
  }
  const unsigned plain = nvc::e4m3_of_magnitude(amax / (6.f * global));
  if (which == 9) return plain > 0 ? plain - 1 : 0;
  if (which == 10) return plain < 126 ? plain + 1 : 126;
  return plain;
}

// The blocks of one buffer of up to 128 columns (cb .. hi - 1), last to first, per launch, 64 matrix rows per workgroup,
// and one wave per scale candidate: the reference's thread walks through its row's candidates one after the other and
// then rounds once more with the winner (src/nvfp4_gpu.hip:66-158); here the ncand waves of a workgroup round the same
// 64 rows at the same time, each under its own candidate, leave their costs in LDS, and the wave whose candidate wins a
// row (smallest cost, the earliest candidate among equals) writes that row's result.  With s the candidate's scale:
//   t_k  = W[k] + F[k] + sum_{j > k in block} d_j L[j][k]       target after the feedback, j ascending
//   q_k  = bf16(level * dec(s) * global)                       what execution sees
//   d_k  = W[k] - q_k                                          error fed back
//   cost = sum_k dw[k] (t_k - q_k)^2                           proxy increment, k descending
// and then F[col] += sum_{j < 16} d_j L[c0 + j][col] (the sum first, in j order, then one add) for the buffer's columns
// left of the block.  Matrix rows do not depend on each other, so a workgroup keeps its rows' F (32 KB) and the block's
// errors in LDS and goes through the blocks without leaving the kernel: bound by the chain of a block's 16 columns
// (4096 x 4096: 32 launches of 64 workgroups, 81 us each, against 480 launches of 10.5 us per block and 7.3 us per
// feedback, 18 us a block with F read and written in memory each time).
// calibrate = 0: no F and no L; the buffers do not depend on each other and blockIdx.y counts them.
// WT: [n][m].  FT: [128][m], the buffer's gathered feedback.  packedT: [n/2][m], scalesT: [n/16][m], ET: [n][m].
constexpr int kBuffer = 128;
__global__ __launch_bounds__(kBlockRows * kScaleTries) void nv_buffer_kernel(
    const float* __restrict__ WT, const float* __restrict__ FT, long m, long n, long cb, const float* __restrict__ L,
    const float* __restrict__ dw, float global, int calibrate, int ncand,
    uint8_t* __restrict__ packedT, uint8_t* __restrict__ scalesT, float* __restrict__ ET) {
  __shared__ __attribute__((aligned(16))) float Lt[16][kBuffer];  // rows c0 .. c0 + 15 of L, columns cb .. c0 + 15
  __shared__ float F[kBuffer][kBlockRows];
  __shared__ float err_lds[16][kBlockRows];
  __shared__ float costs[kScaleTries][kBlockRows];
  const int lane = threadIdx.x & 63;
  const int which = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  cb += long(blockIdx.y) * kBuffer;
  const long hi = n < cb + kBuffer ? n : cb + kBuffer;
  const long r = long(blockIdx.x) * kBlockRows + lane;
  const bool live = r < m;
  if (calibrate) {
    const bool behind = hi < n;  // the last buffer has nothing behind it
    for (int c = which; c < kBuffer; c += ncand) F[c][lane] = behind && live ? FT[c * m + r] : 0.f;
  }
  for (long c0 = hi - 16; c0 >= cb; c0 -= 16) {
    const int left = int(c0 - cb);  // columns of the buffer left of the block
    if (calibrate)
      for (int idx = threadIdx.x; idx < 16 * kBuffer; idx += blockDim.x)
        if ((idx & (kBuffer - 1)) < left + 16)
          Lt[idx / kBuffer][idx & (kBuffer - 1)] = L[(c0 + idx / kBuffer) * n + cb + (idx & (kBuffer - 1))];
    float w[16], t0[16], err[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) w[k] = live ? WT[(c0 + k) * m + r] : 0.f;
    __syncthreads();  // L is there, and F as the block before left it
    float amax = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      t0[k] = w[k] + (calibrate ? F[left + k][lane] : 0.f);
      amax = fmaxf(amax, fabsf(calibrate ? t0[k] : w[k]));
    }
    const unsigned code8 = nv_candidate(which, amax, global);
    const float sd = nvc::e4m3_value(code8);
    const float step = sd * global;
    float cost = 0.f;
    uint32_t nib_lo = 0, nib_hi = 0;  // E2M1 codes of columns 0..7 and 8..15, 4 bits each
#pragma unroll
    for (int k = 15; k >= 0; --k) {
      float t = t0[k];
      if (calibrate) {
#pragma unroll
        for (int j = k + 1; j < 16; ++j) t = fmaf(err[j], Lt[j][left + k], t);
      }
      const float x = step != 0.f ? t / step : 0.f;
      const unsigned mag = nvc::e2m1_of_magnitude(fabsf(x));
      const float q = nvc::through_bf16((x < 0 ? -1.f : 1.f) * nvc::e2m1_value(mag) * sd * global);
      const float weight = dw ? dw[c0 + k] : 1.f;
      cost = fmaf(weight * (t - q), t - q, cost);
      err[k] = w[k] - q;
      const uint32_t nib = mag | ((__float_as_uint(x) >> 31) << 3);
      if (k < 8) nib_lo |= nib << (4 * k);
      else nib_hi |= nib << (4 * (k - 8));
    }
    costs[which][lane] = cost;
    __syncthreads();
    int winner = 0;
    float least = __builtin_inff();
    for (int i = 0; i < ncand; ++i)
      if (costs[i][lane] < least) least = costs[i][lane], winner = i;
    if (winner == which) {
      if (calibrate) {
#pragma unroll
        for (int k = 0; k < 16; ++k) err_lds[k][lane] = err[k];
      }
      if (live) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          packedT[(c0 / 2 + k) * m + r] = uint8_t(nib_lo >> (8 * k));
          packedT[(c0 / 2 + 4 + k) * m + r] = uint8_t(nib_hi >> (8 * k));
        }
        scalesT[(c0 / 16) * m + r] = uint8_t(code8);
        if (calibrate) {
#pragma unroll
          for (int k = 0; k < 16; ++k) ET[(c0 + k) * m + r] = err[k];
        }
      }
    }
    // (also before the costs of the next block, which has no other barrier in front of them when calibrate = 0)
    __syncthreads();
    if (calibrate && left) {
      float e[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) e[j] = err_lds[j][lane];
      for (int c = which; c < left; c += ncand) {
        float acc = 0;
#pragma unroll
        for (int j = 0; j < 16; ++j) acc = fmaf(e[j], Lt[j][c], acc);
        F[c][lane] += acc;
      }
      __syncthreads();  // everyone is through with L before the next block's takes its place
    }
  }
}

// What the matrix's global scale is made from, and whether every value is finite: the largest bit pattern of |w| over the
// matrix (the order of finite magnitudes is that of their bits, and those of infinities and NaNs lie above), one atomic
// maximum per wave.  On one host core this was 9 ms of a 4096 x 4096 call; here 0.11 ms on the copy that is there anyway.
__global__ __launch_bounds__(256) void nv_largest_kernel(const float* __restrict__ w, long count,
                                                         unsigned* __restrict__ top) {
  unsigned most = 0;
  const long step = long(gridDim.x) * 256;
  for (long i = long(blockIdx.x) * 256 + threadIdx.x; i < count; i += step) {
    const unsigned u = __float_as_uint(w[i]) & 0x7fffffffu;
    most = u > most ? u : most;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned o = unsigned(__shfl_xor(int(most), off, 64));
    most = o > most ? o : most;
  }
  if ((threadIdx.x & 63) == 0) atomicMax(top, most);
}
// The feedback a 128-column buffer [cb, cb + 128) receives from every block behind it, gathered in one pass:
//   FT[col - cb][r] = ((0 + a_{n-16}) + a_{n-32}) + ... + a_{cb+128},   a_b = sum_{j < 16} E[b + j][r] * L[b + j][col]
// (each a_b a chain of fused multiply-adds in j order from zero): the values and the order of additions of the
// block-by-block form, which reads and writes every column left of a block once per block (n^2 m / 4 bytes in all);
// this form reads the error rows once per buffer (n^2 m / 64 bytes).  ET: the errors of all finished columns, [n][m].
// A wave: 64 rows x COLS columns; the four waves of a workgroup take four neighbouring column pieces of the same 64 rows,
// so three of them find the error values in the vector L1.  The 16 x COLS piece of L of a block sits in COLS registers,
// row j in lane j of every 16 lanes, and reaches the fused multiply-adds as their broadcast operand (DPP row_newbcast).
// The scalar cache, which brought it before, serves a wave's 16 small pieces per block too slowly.  The values are
// fetched DEPTH - 1 blocks ahead.  Bound by the vector pipes then, one wave per SIMD or a few: 88 us a buffer of a
// 4096 x 4096 matrix on average, 144 before; 248 blocks behind the first buffer take 0.17 ms, 0.34 before.  COLS: 8, or 4
// where 8 would not give every SIMD a wave (m < 4096).
template <int COLS, int DEPTH>
__global__ __launch_bounds__(256) void nv_gather_kernel(float* __restrict__ FT, long m, long n, long cb,
                                                        const float* __restrict__ ET, const float* __restrict__ L) {
  const int lane = threadIdx.x & 63;
  const long row = long(blockIdx.x) * 64 + lane, r = row < m ? row : m - 1;  // no lane leaves: all carry a piece of L
  const long piece = (long(blockIdx.y) * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * COLS;
  float f[COLS], e[DEPTH][16];
  float4 l[DEPTH][COLS / 4];
#pragma unroll
  for (int c = 0; c < COLS; ++c) f[c] = 0.f;
  const float* er = ET + r;
  const float* lr = L + long(lane & 15) * n + cb + piece;
  auto fetch = [&](long b, int s) {
#pragma unroll
    for (int j = 0; j < 16; ++j) e[s][j] = er[(b + j) * m];
#pragma unroll
    for (int c = 0; c < COLS / 4; ++c) l[s][c] = *reinterpret_cast<const float4*>(lr + b * n + 4 * c);
  };
  auto add = [&](int s) {
    float acc[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) acc[c] = 0.f;
    // four j at a time: v_fmac_f32 with the broadcast in its first operand (the compiler does not fold the broadcast into a
    // fused multiply-add by itself); s_nop 1: the wait a vector write of that operand, a copy say, would need before it
#define QTIP_NV_1(ACC, LV, EV, J) \
  "v_fmac_f32_dpp %" #ACC ", %" #LV ", %" #EV " row_newbcast:" #J " row_mask:0xf bank_mask:0xf\n\t"
#define QTIP_NV_4C(EV, J) QTIP_NV_1(0, 4, EV, J) QTIP_NV_1(1, 5, EV, J) QTIP_NV_1(2, 6, EV, J) QTIP_NV_1(3, 7, EV, J)
#define QTIP_NV_4J(C, J0, J1, J2, J3)                                                                                 \
  asm("s_nop 1\n\t" QTIP_NV_4C(8, J0) QTIP_NV_4C(9, J1) QTIP_NV_4C(10, J2) QTIP_NV_4C(11, J3)                         \
      : "+v"(acc[4 * C]), "+v"(acc[4 * C + 1]), "+v"(acc[4 * C + 2]), "+v"(acc[4 * C + 3])                            \
      : "v"(l[s][C].x), "v"(l[s][C].y), "v"(l[s][C].z), "v"(l[s][C].w), "v"(e[s][J0]), "v"(e[s][J1]), "v"(e[s][J2]), \
        "v"(e[s][J3]));
#pragma unroll
    for (int c = 0; c < COLS / 4; ++c) {
      QTIP_NV_4J(c, 0, 1, 2, 3)
      QTIP_NV_4J(c, 4, 5, 6, 7)
      QTIP_NV_4J(c, 8, 9, 10, 11)
      QTIP_NV_4J(c, 12, 13, 14, 15)
    }
#undef QTIP_NV_1
#undef QTIP_NV_4C
#undef QTIP_NV_4J
#pragma unroll
    for (int c = 0; c < COLS; ++c) f[c] += acc[c];
  };
  const long last = cb + kBuffer;
#pragma unroll
  for (int s = 0; s < DEPTH - 1; ++s)
    if (n - 16 - 16 * s >= last) fetch(n - 16 - 16 * s, s);
  for (long b = n - 16; b >= last; b -= 16 * DEPTH) {
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      const long at = b - 16 * s;
      if (at - 16 * (DEPTH - 1) >= last) fetch(at - 16 * (DEPTH - 1), (s + DEPTH - 1) % DEPTH);
      if (at >= last) add(s);
    }
  }
  if (row < m) {
#pragma unroll
    for (int c = 0; c < COLS; ++c) FT[(piece + c) * m + row] = f[c];
  }
}

// bytes [rows][cols] -> [cols][rows], 32 x 32 patches through LDS
__global__ __launch_bounds__(256) void transpose_u8_kernel(const uint8_t* __restrict__ in, long rows, long cols,
                                                           uint8_t* __restrict__ out) {
  __shared__ uint8_t tile[32][33];
  const long r0 = long(blockIdx.y) * 32, c0 = long(blockIdx.x) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long r = r0 + ty + 8 * k, c = c0 + tx;
    tile[ty + 8 * k][tx] = r < rows && c < cols ? in[r * cols + c] : uint8_t(0);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long c = c0 + ty + 8 * k, r = r0 + tx;
    if (c < cols && r < rows) out[c * rows + r] = tile[tx][ty + 8 * k];
  }
}

}  // namespace

void launch_nvfp4_buffer(const float* WT, const float* FT, long m, long n, long cb, const float* L, const float* dw,
                         float global, bool calibrate, bool search, uint8_t* packedT, uint8_t* scalesT, float* ET,
                         hipStream_t s) {
  const int ncand = search ? kScaleTries : 1;
  const dim3 grid(unsigned((m + kBlockRows - 1) / kBlockRows), calibrate ? 1u : unsigned((n + kBuffer - 1) / kBuffer));
  nv_buffer_kernel<<<grid, dim3(unsigned(kBlockRows * ncand)), 0, s>>>(WT, FT, m, n, calibrate ? cb : 0, L, dw, global,
                                                                     calibrate ? 1 : 0, ncand, packedT, scalesT, ET);
  QTIP_HIP(hipGetLastError());
}
void launch_nvfp4_gather(float* FT, long m, long n, long cb, const float* ET, const float* L, hipStream_t s) {
  QTIP_REQUIRE(cb >= 0 && cb % 16 == 0 && cb + kBuffer < n && n % 16 == 0,
               "nvfp4 gather: buffer [%ld, %ld) outside [0, %ld)", cb, cb + kBuffer, n);
  const unsigned rows = unsigned((m + 63) / 64);
  if (m < 4096) nv_gather_kernel<4, 4><<<dim3(rows, kBuffer / 4 / 4), dim3(256), 0, s>>>(FT, m, n, cb, ET, L);
  else nv_gather_kernel<8, 3><<<dim3(rows, kBuffer / 8 / 4), dim3(256), 0, s>>>(FT, m, n, cb, ET, L);
  QTIP_HIP(hipGetLastError());
}
void launch_nvfp4_largest(const float* w, long count, unsigned* top, hipStream_t s) {
  nv_largest_kernel<<<dim3(unsigned(std::min<long>(2048, (count + 255) / 256))), dim3(256), 0, s>>>(w, count, top);
  QTIP_HIP(hipGetLastError());
}
void launch_transpose_u8(const uint8_t* in, long rows, long cols, uint8_t* out, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return;
  transpose_u8_kernel<<<dim3(unsigned((cols + 31) / 32), unsigned((rows + 31) / 32)), dim3(256), 0, s>>>(in, rows, cols, out);
  QTIP_HIP(hipGetLastError());
}

}  // namespace qtipmi
