// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) with true 32-bit arithmetic: products
// and sums on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32,
// IEEE floats in and out, no mode of reduced precision).  It is the matrix
// product of the 32-bit path and the slow, safe product for sizes the other
// kernels refuse.  Numbers below 2^-126 count like any others, in and out.
//
// The order of every sum is fixed by K alone.  k is cut into blocks of 32,
// block b belonging to chain b % 8; half a block (16 products) is summed from
// zero by four instructions, and a chain adds its halves up with the rounding
// errors of the additions collected beside the sum: each exactly where the sum
// so far is the larger of the two, and to the rounding of the half itself where
// it is not (early on, or where the sum is small beside its parts).  At the end
// the eight chains are added, there with the exact error either way, and what
// was collected is taken off.  So a row's result does not depend on the number
// of rows, on the tile it falls in, or on what else is in the batch.  An error that is not finite (a sum
// that has overflowed) is not taken off: infinities stay what they are.
//
// A workgroup is the eight chains of one tile, a wavefront each, operands
// from memory straight into registers.  With few rows the product is bound by
// reading W: eight wavefronts share a tile of 16 columns, so that a narrow W
// (1,024 rows) still keeps 64 compute units loading; one workgroup of 64 x 64
// elements, as this kernel had before, left 16.  With many rows it is bound by
// the matrix cores and by the four vector instructions that every 16 products
// of an element cost behind them, so the tile grows to 32 x 64, for as long as
// there are workgroups for every compute unit.  The next blocks are asked for
// before the products of those at hand, by barriers to the scheduler: left to
// itself it dealt the loads out between the products.  Nothing is asked for
// behind the row's end, except with 32 x 64, where the branch costs more than
// the loads.  Measured with weights from memory, before that in brackets:
// [1024, 3072] at 3 rows 11.1 us (14.4), at 236 26.7 (39.5); [2560, 9728] at
// 8 rows 34.1 us, 2.9 TB/s (42.8), at 700 572, 61 TFLOP/s (575); [6144, 1024]
// at 3 rows 9.3 (11.1); [151936, 1024] at 8 rows 148 us, 4.2 TB/s (160), at
// 236 1,650 (1,773).  (A single chain in workgroups of 64 x 64 elements: 252
// and 408 us for the first, 419 for the last.)
// The error against 64 bits is 7.9e-8 of the result's norm for numbers at
// random (8.1e-8), 2.8e-8 for positive ones (2.8e-8), both at k of 2,048.
//
// Reference counterpart: y = x W^T (+b), W [out, in]
// (crates/prelude-core/src/models/commons/linear.rs:30-98; f32 GEMM with
// 32-bit compute, crates/prelude-cuda/src/ops/gemm.rs:359-365).
#include "common.h"
#include "api.h"

namespace pa {

constexpr int kChains = 8, kBlockK = 32;

struct Eight { f32x4 v[2]; };

// Eight elements of a row from k on; zeros beyond the row's end.  VEC: rows are whole pieces of 16 bytes and k a
// multiple of 8, so the eight are inside or outside together.
template <typename T, bool VEC>
__device__ __forceinline__ Eight load_eight(const T* __restrict__ row, int k, int kk) {
  Eight out;
  if (VEC) {
    const bool in = k < kk;
    const T* at = row + (in ? k : 0);
    if constexpr (sizeof(T) == 4) {
      out.v[0] = *(const f32x4*)at;
      out.v[1] = *(const f32x4*)(at + 4);
    } else {
      const bf16x8 x = *(const bf16x8*)at;
#pragma unroll
      for (int i = 0; i < 8; ++i) out.v[i / 4][i % 4] = (float)x[i];
    }
    if (!in) out.v[0] = out.v[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in = k + i < kk;
      const float x = to_f32(row[in ? k + i : 0]);
      out.v[i / 4][i % 4] = in ? x : 0.f;
    }
  }
  return out;
}

// RM x RN tiles of 16 x 16 a workgroup; D blocks of k loaded at a time, the next D while these are multiplied.
template <typename TA, typename TC, int RM, int RN, int D, bool VEC>
__global__ __launch_bounds__(kChains* kWave) void gemm_plain_kernel(const TA* __restrict__ a, const TA* __restrict__ w,
                                                                    const float* __restrict__ bias, TC* __restrict__ c, int m,
                                                                    int n, int k, long lda, long ldw, long ldc, int act) {
  constexpr int kCols = RN < 2 ? 16 : 32;   // columns added up over the chains at a time
  __shared__ f32x2 sums[kChains][16][kCols];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane % 16, q = lane / 16;
  const int across = (n + 16 * RN - 1) / (16 * RN);
  const int m0 = blockIdx.x / across * 16 * RM, n0 = blockIdx.x % across * 16 * RN;
  const TA* ar[RM];
  const TA* wr[RN];
#pragma unroll
  for (int i = 0; i < RM; ++i) ar[i] = a + (size_t)min(m0 + i * 16 + r, m - 1) * lda;   // rows past the end: any row, not stored
#pragma unroll
  for (int j = 0; j < RN; ++j) wr[j] = w + (size_t)min(n0 + j * 16 + r, n - 1) * ldw;
  f32x4 acc[RM][RN], lost[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = lost[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Operands { Eight a[D][RM], w[D][RN]; };
  auto load = [&](Operands& o, int b) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int at = (b + d * kChains) * kBlockK + q * 8;
#pragma unroll
      for (int j = 0; j < RN; ++j) o.w[d][j] = load_eight<TA, VEC>(wr[j], at, k);
#pragma unroll
      for (int i = 0; i < RM; ++i) o.a[d][i] = load_eight<TA, VEC>(ar[i], at, k);
    }
  };
  auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j) {
            f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              part = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[d][i].v[half][e], o.w[d][j].v[half][e], part, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float t = acc[i][j][e] + part[e];
              lost[i][j][e] += (t - acc[i][j][e]) - part[e];
              acc[i][j][e] = t;
            }
          }
  };
  const int blocks = (k + kBlockK - 1) / kBlockK;
  Operands x, y;
  load(x, wave);
  for (int b = wave; b < blocks; b += 2 * D * kChains) {
    load(y, b + D * kChains);
    __builtin_amdgcn_sched_barrier(0);   // asked for before the products, not between them
    multiply(x);
    if (RM * RN == 8 || b + 2 * D * kChains < blocks) load(x, b + 2 * D * kChains);
    __builtin_amdgcn_sched_barrier(0);
    multiply(y);
  }
  // the chains' sums, 16 rows x kCols columns at a time: lane (r, q) holds column r of rows 4 q .. 4 q + 3
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j0 = 0; j0 < RN; j0 += kCols / 16) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kCols / 16; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[wave][q * 4 + e][j * 16 + r] = f32x2{acc[i][j0 + j][e], lost[i][j0 + j][e]};
      __syncthreads();
      const int row = threadIdx.x / kCols, col = threadIdx.x % kCols;
      const int gm = m0 + i * 16 + row, gn = n0 + j0 * 16 + col;
      if (row < 16 && gm < m && gn < n) {
        f32x2 s = sums[0][row][col];
#pragma unroll
        for (int ch = 1; ch < kChains; ++ch) {
          const f32x2 u = sums[ch][row][col];
          const float t = s[0] + u[0];
          const float back = t - s[0];                       // what was added of u, exactly
          s[1] += u[1] - ((s[0] - (t - back)) + (u[0] - back));
          s[0] = t;
        }
        float v = __builtin_isfinite(s[1]) ? s[0] - s[1] : s[0];
        if (bias) v += bias[gn];
        if (act < 0) {
          c[(size_t)gm * ldc + gn] = from_f32<TC>(v);
        } else {                                               // columns alternate gate_j, up_j (n is even: both are here)
          const float up = __shfl_down(v, 1, kWave);
          if (col % 2 == 0) c[(size_t)gm * ldc + gn / 2] = from_f32<TC>(gate_activation(v, act) * up);
        }
      }
    }
}

template <typename TA, typename TC, int RM, int RN, int D>
int launch_plain_tile(hipStream_t st, bool vec, const TA* a, const TA* w, const float* bias, TC* c, int m, int n, int k, long lda,
                      long ldw, long ldc, int act) {
  const long tiles = (long)((n + 16 * RN - 1) / (16 * RN)) * ((m + 16 * RM - 1) / (16 * RM));
  PA_REQUIRE(tiles <= 0x7fffffffL, "gemm_plain: m=%d and n=%d need %ld workgroups", m, n, tiles);
  const dim3 grid((unsigned)tiles);
  if (vec)
    hipLaunchKernelGGL((gemm_plain_kernel<TA, TC, RM, RN, D, true>), grid, dim3(kChains * kWave), 0, st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  else
    hipLaunchKernelGGL((gemm_plain_kernel<TA, TC, RM, RN, 1, false>), grid, dim3(kChains * kWave), 0, st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  return check_launch("gemm_plain");
}

// Every tile gives the same bits, so the choice is one of speed alone: 16 columns a workgroup where the rows are few and W
// is not so long that workgroups abound; else 32 x 64 where that leaves two workgroups for every compute unit, 32 x 32 where
// that leaves one.
template <typename TA, typename TC>
int launch_plain(hipStream_t st, const void* av, const void* wv, const float* bias, void* cv, int m, int n, int k, long lda,
                 long ldw, long ldc, int act = -1) {
  const TA *a = (const TA*)av, *w = (const TA*)wv;
  TC* c = (TC*)cv;
  constexpr long kPiece = 16 / sizeof(TA);
  const bool vec = k % 8 == 0 && lda % kPiece == 0 && ldw % kPiece == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
  PA_REQUIRE((m + 63) / 64 <= 65535, "gemm_plain: m=%d is more than 64 * 65535 rows", m);   // the face's limit, not the grid's
  auto tiles = [&](long rows, long cols) { return ((m + rows - 1) / rows) * ((n + cols - 1) / cols); };
  if (m <= 16) {
    if (tiles(16, 64) >= 512) return launch_plain_tile<TA, TC, 1, 4, 1>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
    return launch_plain_tile<TA, TC, 1, 1, 2>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  }
  if (tiles(32, 64) >= 512) return launch_plain_tile<TA, TC, 2, 4, 1>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  if (tiles(32, 32) >= 256) return launch_plain_tile<TA, TC, 2, 2, 1>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  return launch_plain_tile<TA, TC, 1, 1, 2>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
}

}  // namespace pa

using namespace pa;

// in_dtype: element type of A and W; out_dtype: element type of C.
extern "C" int pa_gemm_plain(void* stream, int in_dtype, int out_dtype, const void* a, const void* w,
                             const float* bias, void* c, int m, int n, int k, long lda, long ldw, long ldc) {
  if (m == 0 || n == 0) return 0;
  PA_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_plain: bad sizes m=%d n=%d k=%d", m, n, k);
  PA_REQUIRE(lda >= k && ldw >= k && ldc >= n, "gemm_plain: a row stride is smaller than the row (lda=%ld ldw=%ld ldc=%ld)",
             lda, ldw, ldc);
  hipStream_t st = (hipStream_t)stream;
  if (in_dtype == kF32 && out_dtype == kF32) return launch_plain<float, float>(st, a, w, bias, c, m, n, k, lda, ldw, ldc);
  if (in_dtype == kBF16 && out_dtype == kBF16) return launch_plain<bf16, bf16>(st, a, w, bias, c, m, n, k, lda, ldw, ldc);
  if (in_dtype == kBF16 && out_dtype == kF32) return launch_plain<bf16, float>(st, a, w, bias, c, m, n, k, lda, ldw, ldc);
  return pa::fail("gemm_plain: unsupported element types in=%d out=%d", in_dtype, out_dtype);
}

// The same in 32-bit for a weight whose rows alternate gate_j, up_j: C[m, n / 2] = act(gate) * up, the bits of the product and
// pa_silu_mul behind it: a launch of 4.3 us less, and the product's n columns neither written nor read again (28 layers of [6144,
// 1024], a step of 236 rows and five of 3: 15.29 ms before, 14.96 with this).
extern "C" int pa_gemm_plain_gated(void* stream, int act, const void* a, const void* w, void* c, int m, int n, int k, long lda, long ldw, long ldc) {
  if (m == 0 || n == 0) return 0;
  PA_REQUIRE(m > 0 && n > 0 && k > 0 && n % 2 == 0, "gemm_plain_gated: bad sizes m=%d n=%d k=%d", m, n, k);
  PA_REQUIRE(lda >= k && ldw >= k && ldc >= n / 2, "gemm_plain_gated: a row stride is smaller than the row (lda=%ld ldw=%ld ldc=%ld)", lda, ldw, ldc);
  PA_REQUIRE(act == kActSilu || act == kActGeluTanh, "gemm_plain_gated: unknown activation %d", act);
  return launch_plain<float, float>((hipStream_t)stream, a, w, nullptr, c, m, n, k, lda, ldw, ldc, act);
}
