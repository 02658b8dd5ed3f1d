// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) with true 32-bit arithmetic: products
// and sums on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32,
// IEEE floats in and out, no mode of reduced precision).  It is the matrix
// product of the 32-bit path and the slow, safe product for sizes the other
// kernels refuse.  Numbers below 2^-126 count like any others, in and out.
//
// The order of every sum is fixed by K alone.  k is cut into blocks of 32,
// block b belonging to chain b % 8; half a block (16 products) is summed from
// zero by four instructions, and a chain adds its halves up in 64 bits.  At the
// end the eight chains are added, in 64 bits too, and rounded once.  So a row's
// result does not depend on the number of rows, on the tile it falls in, or on
// what else is in the batch.  (With 32-bit sums and the rounding errors of the
// additions collected beside them a number took four instructions of the vector
// ALU where a conversion and an addition are two: [6144, 1024] gated by 150 / 236
// / 2,048 rows 36.6 / 47.1 / 319 us, now 33.6 / 44.3 / 307, [6144, 2560] by 512
// 193 / 183; [1024, 3072] by 236, with 32 x 32 a workgroup, 27.1 / 28.3.)
//
// A workgroup is the eight chains of one tile, a wavefront each, operands
// from memory straight into registers.  (Up to four rows, or eight, and many
// rows of aligned 32-bit operands have kernels of their own below.)  With few
// rows the product is bound by reading W: eight wavefronts share a tile of 16
// columns, so that a narrow W (1,024 rows) still keeps 64 compute units
// loading; one workgroup of 64 x 64 elements, as this kernel had before, left
// 16.  With many rows it is bound by the L2, from which every workgroup reads
// its tile's operands for itself, so the tile grows to 32 x 64, for as long as
// there are workgroups for every compute unit.  The next blocks are asked for
// before the products of those at hand, by barriers to the scheduler: left to
// itself it dealt the loads out between the products.  Nothing is asked for
// behind the row's end, except with 32 x 64, where the branch costs more than
// the loads.  What lies behind the end is made zeros where it is used: in the
// load that was a wait for it, before the products it was to come under.
// Measured with weights from memory: [1024, 3072] at 236 rows 27 us, [1024,
// 2048] 19; [2560, 9728] at 8 rows 34 us, 2.9 TB/s; [151936, 1024] at 8 rows
// 143 us, 4.4 TB/s.
// The error against 64 bits is 7.6e-8 to 7.9e-8 of the result's norm for numbers
// at random, at k of 1,024 to 9,728 and 3 to 2,048 rows (7.7e-8 to 8.0e-8 with
// 32-bit sums).
//
// Reference counterpart: y = x W^T (+b), W [out, in]
// (crates/prelude-core/src/models/commons/linear.rs:30-98; f32 GEMM with
// 32-bit compute, crates/prelude-cuda/src/ops/gemm.rs:359-365).
#include "common.h"
#include "api.h"

namespace pa {

constexpr int kChains = 8, kBlockK = 32;

struct Eight { f32x4 v[2]; };

// Eight elements of a row from k on; beyond the row's end zeros, or, with VEC, any others: rows are whole pieces of 16 bytes
// then and k a multiple of 8, so the eight are inside or outside together, and they are made zeros where they are used (here
// that would wait for the load it has just asked for).
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

typedef double f64x4 __attribute__((ext_vector_type(4)));

// The chains' sums, added in their order and rounded once.
__device__ __forceinline__ float add_chains(const double (&u)[kChains]) {
  double s = u[0];
#pragma unroll
  for (int ch = 1; ch < kChains; ++ch) s += u[ch];
  return (float)s;
}

// Four 32-bit sums onto four of 64 bits.
__device__ __forceinline__ void add_parts(f64x4& acc, f32x4 part) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] += (double)part[e];
}

// RM x RN tiles of 16 x 16 a workgroup; D blocks of k loaded at a time, the next D while these are multiplied.
template <typename TA, typename TC, int RM, int RN, int D, bool VEC>
__global__ __launch_bounds__(kChains* kWave) void gemm_plain_kernel(const TA* __restrict__ a, const TA* __restrict__ w,
                                                                    const float* __restrict__ bias, TC* __restrict__ c, int m,
                                                                    int n, int k, long lda, long ldw, long ldc, int act) {
  constexpr int kCols = RN < 2 ? 16 : 32;   // columns added up over the chains at a time
  __shared__ double sums[kChains][16][kCols];
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
  f64x4 acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = f64x4{0., 0., 0., 0.};
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
  const int blocks = (k + kBlockK - 1) / kBlockK;
  // 32 x 64: four tiles' instructions in turn, so that none waits for the one before, and the adds behind them.  32 x 32: a block that
  // is not there is multiplied all the same, as zeros, rather than branched over ([2048, 6144] by 128 rows 47.8 us, with the branch 49.7,
  // with the other's order too 50.4; 16 x 16 is better off with the branch, 16.9 against 17.1 for [1024, 2048] by 100).
  constexpr bool kLarge = RM * RN == 8, kStraight = RM * RN == 4 && RM == 2;
  constexpr int kJ = kLarge ? 4 / RM : 1;
  auto multiply = [&](Operands& o, int b) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int block = b + d * kChains;
      if (!kStraight && block >= blocks) return;
      if (VEC && block * kBlockK + kBlockK > k && block * kBlockK + q * 8 >= k) {
#pragma unroll
        for (int i = 0; i < RM; ++i) o.a[d][i].v[0] = o.a[d][i].v[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < RN; ++j) o.w[d][j].v[0] = o.w[d][j].v[1] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j0 = 0; j0 < RN; j0 += kJ) {
          f32x4 part[RM][kJ];
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
              for (int j = 0; j < kJ; ++j)
                part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[d][i].v[half][e], o.w[d][j0 + j].v[half][e],
                                                                  e ? part[i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          if (kLarge) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < kJ; ++j) add_parts(acc[i][j0 + j], part[i][j]);
          if (kLarge) __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  Operands x, y;
  load(x, wave);
  for (int b = wave; b < blocks; b += 2 * D * kChains) {
    load(y, b + D * kChains);
    __builtin_amdgcn_sched_barrier(0);   // asked for before the products, not between them
    multiply(x, b);
    if (kLarge || b + 2 * D * kChains < blocks) load(x, b + 2 * D * kChains);
    __builtin_amdgcn_sched_barrier(0);
    multiply(y, b + D * kChains);
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
        for (int e = 0; e < 4; ++e) sums[wave][q * 4 + e][j * 16 + r] = acc[i][j0 + j][e];
      __syncthreads();
      const int row = threadIdx.x / kCols, col = threadIdx.x % kCols;
      const int gm = m0 + i * 16 + row, gn = n0 + j0 * 16 + col;
      if (row < 16 && gm < m && gn < n) {
        double u[kChains];
#pragma unroll
        for (int ch = 0; ch < kChains; ++ch) u[ch] = sums[ch][row][col];
        float v = add_chains(u);
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

// The same sums, bit for bit, for a few rows.  v_mfma_f32_16x16x4_f32 adds its four products one after the other with an fma's
// rounding each, and v_mfma_f32_4x4x1_f32, sixteen products of 4 x 1 by 1 x 4, rounds as an fma does: given the numbers in the
// same order of k it gives the same sums, of four rows in place of sixteen.
//
// A workgroup owns eight columns: the sixteen small matrices are two groups of four columns by the eight chains.  k is cut into
// pieces of 256, the eight chains' next block each; a wavefront takes every `waves`-th piece for itself, from memory into LDS
// without registers in between, the first of all wavefronts on their way at once, and leaves the halves' sums in LDS, where 256
// threads (row, column, chain) add them up in their order.
//
// What bounds it is the way of W to the compute units, of which a narrow weight gets few, and beside that LDS reads and the
// length of the path: a piece is sixteen reads and 32 matrix instructions whatever the number of rows (a row a wavefront on the
// vector ALU, each reading W for itself: 64 reads a piece, 0.7 us).  With weights from memory, at 3 rows, in us (16 columns a
// workgroup and the 16-row instruction / this): [1024, 1024] 5.2 / 3.9, [1024, 3072] 11.0 / 6.7, [4096, 1024] 6.6 / 6.1, [6144, 1024]
// 9.1 / 7.4, [2560, 9728] 33.4 / 26.2, [6144, 2560] 20.4 / 16.1, [151936, 1024] 140 / 110 (5.7 TB/s).
constexpr int kFewCols = 8, kFewPieceK = kChains * kBlockK;
// Five to eight rows are two groups of four, and more LDS a piece, which leaves wide weights fewer workgroups a compute unit: at 8
// rows [1024, 3072] 12.3 / 8.1, [2048, 2048] 9.4 / 7.4, [2048, 6144] 21.7 / 14.8, but [4096, 1024] 6.8 / 7.0, [2560, 4096] 16.0 / 21.0.
constexpr int kFewEightMostN = 2048;
constexpr unsigned kFewLds = 150 * 1024;

__device__ __forceinline__ void few_load(const float* src, unsigned lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) unsigned*)src,
                                   (__attribute__((address_space(3))) unsigned*)lds, 16, 0, 0);
}

// Where the 16-byte pieces of chain h of row or column c lie within its kilobyte: piece p at 8 h + (p ^ few_turn), so that sixteen
// lanes reading piece p of four chains and four columns, neighbours or two apart, find it in as many different banks.
__device__ __forceinline__ int few_turn(int h, int c) { return (c & 3) | (((h >> 1) ^ (h >> 2)) & 1) << 2; }

// A lane's 32 numbers of a piece, at `at` ^ 16 p.  One block of assembly with its own wait: LDS that loads write behind the
// compiler's back is read in a known place, and no register is handed on before it is there.
__device__ __forceinline__ void few_read(f32x4 (&v)[8], unsigned at) {
  asm volatile(
      "ds_read_b128 %0, %8\nds_read_b128 %1, %9\nds_read_b128 %2, %10\nds_read_b128 %3, %11\nds_read_b128 %4, %12\n"
      "ds_read_b128 %5, %13\nds_read_b128 %6, %14\nds_read_b128 %7, %15\ns_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(at), "v"(at ^ 16), "v"(at ^ 32), "v"(at ^ 48), "v"(at ^ 64), "v"(at ^ 80), "v"(at ^ 96), "v"(at ^ 112)
      : "memory");
}
__device__ __forceinline__ void few_read(f32x4 (&v)[8], f32x4 (&w)[8], unsigned at, unsigned bt) {
  asm volatile(
      "ds_read_b128 %0, %16\nds_read_b128 %8, %24\nds_read_b128 %1, %17\nds_read_b128 %9, %25\n"
      "ds_read_b128 %2, %18\nds_read_b128 %10, %26\nds_read_b128 %3, %19\nds_read_b128 %11, %27\n"
      "ds_read_b128 %4, %20\nds_read_b128 %12, %28\nds_read_b128 %5, %21\nds_read_b128 %13, %29\n"
      "ds_read_b128 %6, %22\nds_read_b128 %14, %30\nds_read_b128 %7, %23\nds_read_b128 %15, %31\ns_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
        "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7])
      : "v"(at), "v"(at ^ 16), "v"(at ^ 32), "v"(at ^ 48), "v"(at ^ 64), "v"(at ^ 80), "v"(at ^ 96), "v"(at ^ 112),
        "v"(bt), "v"(bt ^ 16), "v"(bt ^ 32), "v"(bt ^ 48), "v"(bt ^ 64), "v"(bt ^ 80), "v"(bt ^ 96), "v"(bt ^ 112)
      : "memory");
}

// The rows that a product of few rows norms for itself before it multiplies them: res + x (written to res_out by the first workgroup)
// over its root mean square, times gain, in rmsnorm_vec_kernel's order to the bit: a wavefront's piece of 256 is what a wavefront has there.
template <bool NORMED> struct FewNorm {};
template <> struct FewNorm<true> {
  const float *res, *gain;
  float* res_out;
  float eps;
};

// RG groups of four rows.  k in whole blocks of 32.  LDS: a piece a wavefront (eight columns and 4 RG rows, 1 KB each); the halves'
// sums take their place where every wavefront has one piece, else two places a wavefront of their own (`parts` from there on).
//
// NORMED (a piece a wavefront, rows of a beside each other): the add and the norm in front of the product, by every workgroup for
// itself while its weight is on the way, in place of a launch: what is added to the path is a trip to the L2, the sums over the
// wavefronts and one pass through LDS.  [4096, 1024] at 3 rows in a chain, us: 8.4 apart, 6.9 like this (7.8 with a row's sums, and its
// root, one after the other); [6144, 1024] gated 9.5 / 8.2.
template <int RG, bool NORMED>
__global__ __launch_bounds__(12 * kWave) void gemm_plain_few_kernel(
    const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ c, int m, int n, int k,
    long lda, long ldw, long ldc, int act, FewNorm<NORMED> norm) {
  extern __shared__ __align__(128) unsigned char lds_raw[];
  __shared__ double sums[4 * RG][kFewCols][kChains + 1];
  constexpr int kPiece = (kFewCols + 4 * RG) * 1024, kPart = 4 * RG * kFewCols * kChains;   // bytes; pairs of 32-bit numbers
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_raw;
  const int waves = blockDim.x / kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int n0 = blockIdx.x * kFewCols, pieces = (k + kFewPieceK - 1) / kFewPieceK;
  const bool once = pieces <= waves;
  // what the lane fetches of row or column j of a piece: 16 bytes of chain lane / 8, which of them goes by j % 4
  const int fetched = lane / 8;
  auto ask = [&](int p) {
    const int k0 = p * kFewPieceK + fetched * kBlockK;
    const int from = k0 < k ? k0 : 0;                             // chains without a block here: any numbers, not used
    const unsigned at = lds + wave * kPiece;
#pragma unroll
    for (int j = 0; j < (NORMED ? kFewCols : kFewCols + 4 * RG); ++j) {
      const float* row = j < kFewCols ? w + (size_t)min(n0 + j, n - 1) * ldw : a + (size_t)min(j - kFewCols, m - 1) * lda;
      few_load(row + from + ((lane % 8) ^ few_turn(fetched, j)) * 4, at + j * 1024);   // rows and columns past the end: any that exist
    }
  };
  f32x4 sum[NORMED ? 4 * RG : 1];
  const int mine = wave * kFewPieceK + lane * 4;                  // the lane's four numbers of a row that is normed here
  if constexpr (NORMED) {
    __shared__ float squares[12][4 * RG];
    const size_t from = mine < k ? mine : 0;
    f32x4 r[4 * RG];
#pragma unroll
    for (int j = 0; j < 4 * RG; ++j) {
      const size_t at = (size_t)min(j, m - 1) * k + from;
      sum[j] = *reinterpret_cast<const f32x4*>(a + at), r[j] = *reinterpret_cast<const f32x4*>(norm.res + at);
    }
    const f32x4 gain = *reinterpret_cast<const f32x4*>(norm.gain + from);
    __builtin_amdgcn_sched_barrier(0);
    ask(wave < pieces ? wave : 0);
    __builtin_amdgcn_sched_barrier(0);
    float ss[4 * RG];
#pragma unroll
    for (int j = 0; j < 4 * RG; ++j) {
      ss[j] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sum[j][e] += r[j][e];
        ss[j] += sum[j][e] * sum[j][e];
      }
      ss[j] = wave_sum(mine < k ? ss[j] : 0.f);
    }
    float own = ss[0];
#pragma unroll
    for (int j = 1; j < 4 * RG; ++j) own = lane == j ? ss[j] : own;
    if (lane < 4 * RG) squares[wave][lane] = own;
    asm volatile("s_waitcnt lgkmcnt(0)\ns_barrier" ::: "memory");
    float parts[12], total = 0.f;                                 // a row a lane, all read at once, added in the wavefronts' order
#pragma unroll
    for (int i = 0; i < 12; ++i) parts[i] = squares[i][lane % (4 * RG)];
#pragma unroll
    for (int i = 0; i < 12; ++i) total += i < pieces ? parts[i] : 0.f;
    const float inv = rsqrtf(total / (float)k + norm.eps);
    unsigned char* const rows = lds_raw + wave * kPiece + kFewCols * 1024;
#pragma unroll
    for (int j = 0; j < 4 * RG; ++j) {
      const float row_inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), j));
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = sum[j][e] * row_inv * gain[e];
      *reinterpret_cast<f32x4*>(rows + j * 1024 + fetched * 128 + ((lane % 8) ^ few_turn(fetched, j)) * 16) = v;
    }
  } else {
    ask(wave < pieces ? wave : 0);
  }
  // lane (matrix lane / 4, place lane % 4): chain h, column col, and row lane % 4 of A
  const int h = lane / 4 % 8, col = lane / 32 * 4 + lane % 4;
  const unsigned turned = lds + wave * kPiece + h * 128 + few_turn(h, lane) * 16;
  // the additions: four wavefronts, a thread the column ac and chain ah of the rows ar, ar + 4
  const int ah = threadIdx.x % kChains, ac = threadIdx.x / kChains % kFewCols, ar = wave;
  double acc[RG] = {};
  for (int p0 = 0, round = 0; p0 < pieces; p0 += waves, ++round) {
    auto parts_of = [&](int v) {
      return reinterpret_cast<f32x2*>(lds_raw + (once ? v * kPiece : waves * kPiece + ((round & 1) * waves + v) * kPart * 8));
    };
    const int p = p0 + wave;
    if (p < pieces) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // the wavefront's own loads: nobody else reads them
      f32x4 wv[8], av[RG][8];
      few_read(wv, av[0], turned + col * 1024, turned + (kFewCols + lane % 4) * 1024);
#pragma unroll
      for (int i = 1; i < RG; ++i) few_read(av[i], turned + (kFewCols + 4 * i + lane % 4) * 1024);
      if (p + waves < pieces) ask(p + waves);
      f32x2* out = parts_of(wave);
#pragma unroll
      for (int i = 0; i < RG; ++i) {
        f32x4 part[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int e = 0; e < 4; ++e)                               // the larger instruction's order: its four k, 8 apart, then the next four
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int half = 0; half < 2; ++half)
              part[half] = __builtin_amdgcn_mfma_f32_4x4x1f32(av[i][q * 2 + half][e], wv[q * 2 + half][e], part[half], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[((i * 4 + e) * kFewCols + col) * kChains + h] = f32x2{part[0][e], part[1][e]};
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\ns_barrier" ::: "memory");
    const int here = min(waves, pieces - p0);
    if (ar < 4) {
      for (int v = 0; v < here; ++v) {
        const f32x2* parts = parts_of(v);
        const bool in = (p0 + v) * kFewPieceK + ah * kBlockK < k;
#pragma unroll
        for (int i = 0; i < RG; ++i) {
          const f32x2 part = parts[i * 4 * kFewCols * kChains + threadIdx.x];
#pragma unroll
          for (int half = 0; half < 2; ++half) acc[i] += in ? (double)part[half] : 0.;
        }
      }
    }
  }
  if constexpr (NORMED) {
    if (blockIdx.x == 0 && mine < k) {
#pragma unroll
      for (int j = 0; j < 4 * RG; ++j)
        if (j < m) *reinterpret_cast<f32x4*>(norm.res_out + (size_t)j * k + mine) = sum[j];
    }
  }
  if (ar < 4) {
#pragma unroll
    for (int i = 0; i < RG; ++i) sums[i * 4 + ar][ac][ah] = acc[i];
  }
  __syncthreads();
  if ((int)threadIdx.x >= 4 * RG * kFewCols) return;               // a row's eight columns are neighbours, within one wavefront
  const int row = threadIdx.x / kFewCols, gn = n0 + threadIdx.x % kFewCols;
  double u[kChains];
#pragma unroll
  for (int ch = 0; ch < kChains; ++ch) u[ch] = sums[row][threadIdx.x % kFewCols][ch];
  float v = add_chains(u);
  if (bias) v += bias[min(gn, n - 1)];
  const float up = act < 0 ? 0.f : __shfl_down(v, 1, kWave);
  if (row >= m || gn >= n) return;
  if (act < 0) c[(size_t)row * ldc + gn] = v;
  else if (gn % 2 == 0) c[(size_t)row * ldc + gn / 2] = gate_activation(v, act) * up;
}

template <int RG>
struct FewPlan {   // wavefronts a workgroup and its LDS
  static constexpr unsigned kPiece = (kFewCols + 4 * RG) * 1024, kParts = 2 * 4 * RG * kFewCols * kChains * 8;
  int waves;
  unsigned bytes;
  FewPlan(int n, int k) {
    const int pieces = (k + kFewPieceK - 1) / kFewPieceK, groups = (n + kFewCols - 1) / kFewCols;
    // a wavefront a piece where one workgroup, or the two or three that a compute unit then gets, have LDS for that many ([2560, 9728]
    // 26.2 us with four wavefronts a workgroup, two workgroups a compute unit); else as many as have room
    const unsigned room = kFewLds / (groups <= 256 ? 1 : (groups <= 512 ? 2 : 3));
    waves = pieces;
    bytes = pieces * kPiece;
    if (pieces > 12 || bytes > room) {
      waves = room / (kPiece + kParts);
      waves = waves < 4 ? 4 : (waves < 12 ? waves : 12);
      bytes = waves * (kPiece + kParts);
    }
    if (waves < 4) waves = 4, bytes = waves * kPiece;             // the additions' threads
  }
};

template <int RG, bool NORMED = false>
int launch_plain_few(hipStream_t st, const float* a, const float* w, const float* bias, float* c, int m, int n, int k, long lda, long ldw,
                     long ldc, int act, FewNorm<NORMED> norm = {}) {
  static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_plain_few_kernel<RG, NORMED>),
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds);
  if (allowed != hipSuccess) return pa::fail("gemm_plain: %u bytes of LDS refused: %s", kFewLds, hipGetErrorString(allowed));
  const FewPlan<RG> plan(n, k);
  hipLaunchKernelGGL((gemm_plain_few_kernel<RG, NORMED>), dim3((n + kFewCols - 1) / kFewCols), dim3(plan.waves * kWave), plan.bytes, st, a, w,
                     bias, c, m, n, k, lda, ldw, ldc, act, norm);
  return check_launch("gemm_plain");
}

// The same sums, bit for bit, for many rows, in whole blocks of 32 of aligned 32-bit operands.  A wavefront owns TM x TN tiles of the
// result and goes through the chains one after the other, so that it holds one chain's sum and the sum of those before it; operands
// pass through LDS, S stages of one block of k.  KS groups of wavefronts share the chains of the same tiles between them.
//
// What bounds it is each SIMD's instructions: a tile is 8 instructions of the matrix cores of 32 cycles and 16 of the vector ALU, half of them
// additions of 64 bits, a block, and the two do not overlap, neither in one wavefront (dealt out one to four) nor in two half a step apart.
// Beside that, the reads of LDS and the barrier of a block, which other workgroups of the
// compute unit cover.  With 32-bit sums, 32 instructions (48 cycles for 1,024 products, 105 TFLOP/s at most), against the kernel
// above, whose eight wavefronts each read the whole tile's operands from the L2: [6144, 1024] at 150 / 236 / 450 / 2,048 rows 33.4 /
// 45.4 / 81.4 / 302 us where it took 41.0 / 53.4 / 100 / 397, [4096, 1024] at 450 55.5 (68.6), [6144, 2560] at 512 188 (210), [1024,
// 3072] at 300 46.6 (50.4), but at 236 30.3 (26.0).
template <int TM, int TN>
__device__ __forceinline__ void rows_read(f32x4 (&a)[TM][2], f32x4 (&w)[TN][2], unsigned at, unsigned wt) {
  // one block of assembly with its own wait, as for few rows
  if constexpr (TM == 2 && TN == 1)
    asm volatile(
        "ds_read_b128 %0, %6\nds_read_b128 %4, %8\nds_read_b128 %2, %6 offset:2048\n"
        "ds_read_b128 %1, %7\nds_read_b128 %5, %9\nds_read_b128 %3, %7 offset:2048\ns_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(w[0][0]), "=&v"(w[0][1])
        : "v"(at), "v"(at ^ 16), "v"(wt), "v"(wt ^ 16)
        : "memory");
  else {
    static_assert(TM == 1 && TN == 1);
    asm volatile("ds_read_b128 %0, %4\nds_read_b128 %2, %6\nds_read_b128 %1, %5\nds_read_b128 %3, %7\ns_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(w[0][0]), "=&v"(w[0][1])
                 : "v"(at), "v"(at ^ 16), "v"(wt), "v"(wt ^ 16)
                 : "memory");
  }
}

template <int WM, int WN, int TM, int TN, int KS, int S>
struct RowsShape {
  static constexpr int kRows = 16 * WM * TM, kCols = 16 * WN * TN, kGroup = WM * WN, kUnits = (kRows + kCols) / 8;
  static constexpr int kThreads = kGroup * KS * kWave, kStage = KS * kUnits * 1024, kLds = S * kStage;
};

template <int WM, int WN, int TM, int TN, int KS, int S>
__global__ __launch_bounds__(WM* WN* KS* kWave) void gemm_plain_rows_kernel(
    const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ c, int m, int n, int k,
    long lda, long ldw, long ldc, int act) {
  typedef RowsShape<WM, WN, TM, TN, KS, S> Shape;
  constexpr int kGroup = Shape::kGroup, kLoads = (Shape::kUnits + kGroup - 1) / kGroup, kOwn = kChains / KS;   // chains a group
  extern __shared__ __align__(128) unsigned char lds_raw[];
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_raw;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int group = wave / kGroup, gw = wave % kGroup, wm = gw / WN, wn = gw % WN;
  const int across = (n + Shape::kCols - 1) / Shape::kCols;
  const int m0 = blockIdx.x / across * Shape::kRows, n0 = blockIdx.x % across * Shape::kCols;
  const int blocks = k / kBlockK;
  // A stage is a kilobyte for every eight rows of A and W (W's behind A's); 16-byte piece p of row r lies at 8 r + (p ^ r / 2 % 8), so
  // that sixteen rows' pieces p are in as many different banks.  The group's wavefronts ask for every kGroup-th kilobyte.
  const int turn = (gw % 2 * 4 + lane / 16) % 8;
  const float* src[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = (gw + i * kGroup) * 8 + lane / 8;               // (rows and columns past the end: the last one)
    src[i] = (row < Shape::kRows ? a + (size_t)min(m0 + row, m - 1) * lda : w + (size_t)min(n0 + row - Shape::kRows, n - 1) * ldw) +
             ((lane % 8) ^ turn) * 4;
  }
  const bool all = Shape::kUnits % kGroup == 0 || gw < Shape::kUnits % kGroup;   // it asks kLoads times, else once less
  int ask_ch = group * kOwn, ask_b = ask_ch, stage_at = 0;
  auto ask = [&]() {
    const int at = ask_ch < (group + 1) * kOwn && ask_b < blocks ? ask_b * kBlockK : 0;   // behind the last block: any, not used
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      if (i + 1 < kLoads || all) few_load(src[i] + at, lds + stage_at + (group * Shape::kUnits + gw + i * kGroup) * 1024);
    ask_b += kChains;
    if (ask_b >= blocks) ask_b = ++ask_ch;
    stage_at = stage_at + Shape::kStage == Shape::kLds ? 0 : stage_at + Shape::kStage;
  };
  int steps = 0;                                                    // the first group's, which has the most
#pragma unroll
  for (int ch = 0; ch < kOwn; ++ch) steps += ch < blocks ? (blocks - ch + kChains - 1) / kChains : 0;
#pragma unroll
  for (int i = 0; i < S - 1; ++i) ask();
  const int r = lane % 16, q = lane / 16;
  const unsigned inner = r * 128 + ((2 * q) ^ (r / 2)) * 16 + lds + group * Shape::kUnits * 1024;
  const unsigned at0 = inner + wm * TM * 2048, wt0 = inner + Shape::kRows * 128 + wn * TN * 2048;
  f64x4 acc[TM][TN] = {};
  constexpr int kKept = KS == 1 ? 1 : kOwn;                         // the first group keeps the sum of its chains, the others each chain's
  f64x4 sum[kKept][TM][TN] = {};
  int ch = group * kOwn, b = ch, read_at = 0;
  for (int step = 0; step < steps; ++step) {
    if (all) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads * (S - 2)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kLoads - 1) * (S - 2)) : "memory");
    asm volatile("s_barrier" ::: "memory");                         // this stage is there; the one before is read by all
    ask();
    const int stage = read_at;
    read_at = read_at + Shape::kStage == Shape::kLds ? 0 : read_at + Shape::kStage;
    if (ch >= (group + 1) * kOwn || b >= blocks) continue;
    f32x4 av[TM][2], wv[TN][2];
    rows_read<TM, TN>(av, wv, at0 + stage, wt0 + stage);
    f32x4 part[2][TM][TN];
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            part[half][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i][half][e], wv[j][half][e],
                                                                    e ? part[half][i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) add_parts(acc[i][j], part[half][i][j]);
    b += kChains;
    if (b < blocks) continue;
    if (group == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[0][i][j] += acc[i][j];
    } else {
#pragma unroll
      for (int o = 0; o < kKept; ++o)
        if (ch - group * kOwn == o) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) sum[o][i][j] = acc[i][j];
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f64x4{0., 0., 0., 0.};
    b = ++ch;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // what was asked for behind the end goes to LDS too
  if constexpr (KS > 1) {                                           // the other groups' chains, in their order
    f64x4* place = reinterpret_cast<f64x4*>(lds_raw) + gw * kWave + lane;
#pragma unroll
    for (int g = 1; g < KS; ++g)
#pragma unroll
      for (int o = 0; o < kKept; ++o) {
        __syncthreads();
        if (group == g)
#pragma unroll
          for (int t = 0; t < TM * TN; ++t) place[t * kGroup * kWave] = sum[o][t / TN][t % TN];
        __syncthreads();
        if (group == 0)
#pragma unroll
          for (int t = 0; t < TM * TN; ++t) sum[0][t / TN][t % TN] += place[t * kGroup * kWave];
      }
    if (group) return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int gn = n0 + (wn * TN + j) * 16 + r;
    const float plus = bias ? bias[min(gn, n - 1)] : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int gm = m0 + (wm * TM + i) * 16 + q * 4 + e;
        float v = (float)sum[0][i][j][e];
        if (bias) v += plus;
        if (act < 0) {
          if (gm < m && gn < n) c[(size_t)gm * ldc + gn] = v;
        } else {                                                    // columns alternate gate_j, up_j (n is even)
          const float up = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xf5, 0xf, 0xf, true));   // one lane on
          if (gm < m && gn < n && r % 2 == 0) c[(size_t)gm * ldc + gn / 2] = gate_activation(v, act) * up;
        }
      }
  }
}

template <int WM, int WN, int TM, int TN, int KS, int S>
int launch_plain_rows(hipStream_t st, const float* a, const float* w, const float* bias, float* c, int m, int n, int k, long lda, long ldw,
                      long ldc, int act) {
  typedef RowsShape<WM, WN, TM, TN, KS, S> Shape;
  const auto kernel = &gemm_plain_rows_kernel<WM, WN, TM, TN, KS, S>;
  static const hipError_t allowed =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kLds);
  if (allowed != hipSuccess) return pa::fail("gemm_plain: %d bytes of LDS refused: %s", (int)Shape::kLds, hipGetErrorString(allowed));
  const long tiles = (long)((n + Shape::kCols - 1) / Shape::kCols) * ((m + Shape::kRows - 1) / Shape::kRows);
  PA_REQUIRE(tiles <= 0x7fffffffL, "gemm_plain: m=%d and n=%d need %ld workgroups", m, n, tiles);
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(Shape::kThreads), Shape::kLds, st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
  return check_launch("gemm_plain");
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

// What a product of more than sixteen rows of whole blocks of aligned 32-bit operands is priced at, in us, in workgroups of rows x
// cols: `fixed`, and every block of k the first workgroup of a compute unit, the second, and each one more.  Fitted to [1024, 2048],
// [1024, 3072], [4096, 1024] and [6144, 1024] at 40 to 450 rows and the weights of hidden 2,560 at 512, with weights from memory: over
// sixteen weights of 768 to 19,456 rows and 768 to 9,728 columns by 17 to 2,048 rows the choice takes more than 3 % longer than the
// fastest in 21 of 256 products, 9 % at most ([19456, 2560] by 1,024 rows 1,210 us in 32 x 64, 1,114 in 64 x 64).  Workgroups of 16 x 16
// read too much from the L2 where there are many.
enum PlainShape { kPlain16x16, kPlain32x32, kRows32x32, kRows32x64, kRows64x64 };
struct PlainPrice {
  PlainShape shape;
  int rows, cols;
  double fixed, first, second, more;
  double of(int m, int n, int k) const {
    const long tiles = (long)((m + rows - 1) / rows) * ((n + cols - 1) / cols), each = (tiles + 255) / 256;
    if (shape == kPlain16x16 && each > 2) return 1e30;
    return fixed + k / kBlockK * (first + (each > 1 ? second : 0.0) + (each > 2 ? (each - 2) * more : 0.0));
  }
};
constexpr PlainPrice kPlainPrices[] = {{kPlain32x32, 32, 32, 5.0, 0.228, 0.27, 0.285},
                                       {kPlain16x16, 16, 16, 2.3, 0.122, 0.105, 0.105},
                                       {kRows32x32, 32, 32, 5.2, 0.275, 0.18, 0.265},
                                       {kRows32x64, 32, 64, 4.2, 0.56, 0.34, 0.39},
                                       {kRows64x64, 64, 64, 5.5, 0.87, 0.68, 0.8}};

// Every tile gives the same bits, so the choice is one of speed alone: by price where the operands allow all; else 16 columns a
// workgroup where the rows are few and W is not so long that workgroups abound; else 32 x 64 where that leaves two workgroups for
// every compute unit, 32 x 32 where that leaves one.
template <typename TA, typename TC>
int launch_plain(hipStream_t st, const void* av, const void* wv, const float* bias, void* cv, int m, int n, int k, long lda,
                 long ldw, long ldc, int act = -1) {
  const TA *a = (const TA*)av, *w = (const TA*)wv;
  TC* c = (TC*)cv;
  constexpr long kPiece = 16 / sizeof(TA);
  const bool vec = k % 8 == 0 && lda % kPiece == 0 && ldw % kPiece == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
  PA_REQUIRE((m + 63) / 64 <= 65535, "gemm_plain: m=%d is more than 64 * 65535 rows", m);   // the face's limit, not the grid's
  auto tiles = [&](long rows, long cols) { return ((m + rows - 1) / rows) * ((n + cols - 1) / cols); };
  if constexpr (sizeof(TA) == 4 && sizeof(TC) == 4) {
    if (vec && k % kBlockK == 0) {
      if (m <= 4) return launch_plain_few<1>(st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
      if (m <= 8 && n <= kFewEightMostN) return launch_plain_few<2>(st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
      if (m > 16) {
        PlainPrice best = kPlainPrices[0];
        for (const PlainPrice& p : kPlainPrices)
          if (p.of(m, n, k) < best.of(m, n, k)) best = p;
        switch (best.shape) {
          case kPlain16x16: return launch_plain_tile<TA, TC, 1, 1, 2>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
          case kPlain32x32: return launch_plain_tile<TA, TC, 2, 2, 1>(st, vec, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
          case kRows32x32: return launch_plain_rows<2, 2, 1, 1, 2, 4>(st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
          case kRows32x64: return launch_plain_rows<2, 4, 1, 1, 1, 4>(st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
          case kRows64x64: return launch_plain_rows<2, 4, 2, 1, 1, 4>(st, a, w, bias, c, m, n, k, lda, ldw, ldc, act);
        }
      }
    }
  }
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

// Whether pa_gemm_plain_normed takes a product of m rows by [n, k]: by gemm_plain_few_kernel, a piece a wavefront.
extern "C" int pa_gemm_plain_normed_takes(int m, int n, int k) {
  if (m < 1 || n < 1 || k < kBlockK || k % kBlockK || m > 8 || (m > 4 && n > kFewEightMostN)) return 0;
  return (m <= 4 ? FewPlan<1>(n, k).waves : FewPlan<2>(n, k).waves) * kFewPieceK >= k;
}

// C = f(h W^T (+ bias)) for h = rmsnorm(res + x; gain, eps) of a few rows in 32-bit, res_out = res + x: pa_rmsnorm and pa_gemm_plain
// (act -1) or pa_gemm_plain_gated in one launch, to the bit.  x, res and res_out [m, k], w [n, k]; res_out is neither x nor res.
extern "C" int pa_gemm_plain_normed(void* stream, int act, const float* x, const float* res, const float* gain, float eps, float* res_out,
                                    const float* w, const float* bias, float* c, int m, int n, int k, long ldc) {
  if (m == 0 || n == 0) return 0;
  PA_REQUIRE(pa_gemm_plain_normed_takes(m, n, k), "gemm_plain_normed: sizes m=%d n=%d k=%d are not taken", m, n, k);
  PA_REQUIRE(x && res && gain && res_out && w && c, "gemm_plain_normed: an operand is missing");
  PA_REQUIRE(res_out != res && res_out != x, "gemm_plain_normed: the new residual needs a buffer of its own");
  PA_REQUIRE((((uintptr_t)x | (uintptr_t)res | (uintptr_t)gain | (uintptr_t)res_out | (uintptr_t)w) & 15) == 0,
             "gemm_plain_normed: operands are not 16-byte aligned");
  PA_REQUIRE(act == -1 || act == kActSilu || act == kActGeluTanh, "gemm_plain_normed: unknown activation %d", act);
  PA_REQUIRE(act < 0 || (n % 2 == 0 && !bias), "gemm_plain_normed: the gated epilogue needs an even n and no bias");
  PA_REQUIRE(ldc >= (act < 0 ? n : n / 2), "gemm_plain_normed: output row stride %ld is too small", ldc);
  const FewNorm<true> norm{res, gain, res_out, eps};
  if (m <= 4) return launch_plain_few<1, true>((hipStream_t)stream, x, w, bias, c, m, n, k, k, k, ldc, act, norm);
  return launch_plain_few<2, true>((hipStream_t)stream, x, w, bias, c, m, n, k, k, k, ldc, act, norm);
}
