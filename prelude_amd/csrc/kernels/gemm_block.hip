// C[M,N] = X[M,K] * W[N,K]^T for many rows in bfloat16 with 32-bit accumulation, from the weight in tiles (pa_pack_tiles),
// both operands through LDS (block_core.h): prompts, and batches beyond what gemm_mid.hip takes.
//
// Workgroups of several shapes, from 256 x 256 outputs for products that fill the chip several times over to 64 x 64 for 128
// rows of a small model; K may be cut into slices whose 32-bit partial sums the reader adds (the residual add + RMSNorm kernel
// does as it loads).  Which shape and how many slices is priced by what was measured of each (block_shapes).  The tiles
// that share rows of W or of X get consecutive places on one XCD.
//
// Epilogues: bfloat16 out (+ bias); act(gate) * up over rows that alternate gate_j, up_j; the clamped gated pair; the
// square of relu; the slices.  The activations are computed in 32-bit of unrounded sums with the hardware's exponential and
// reciprocal: behind the rounding to bfloat16 the distance from 64-bit is that of expf, tanhf and a division to ten digits, and
// those take 4 to 9 % of the product ([19456, 2560] by 2,048 rows 187 us against 172, [16384, 2048] 124 against 111).
//
// Measured inside a graph with weights from memory, against the library's product (and the activation kernel behind it where
// the product is gated), in us: [19456, 2560] gated by 2,048 rows 160 against 225 (by 512 rows 50 against 65), [6144, 2560]
// 50 against 59, [24576, 4096] gated by 1,531 rows 221 against 278, [6144, 4096] 63 against 76; in slices [2560, 9728] by 2,048
// rows 78 against 108 (by 512 rows 30 against 51), [4096, 12288] by 1,531 rows 119 against 147; by 128 rows [4096, 1024] 6.3
// against 9.0, [1024, 3072] in four slices 5.7 against 7.9.
//
// Reference counterpart: the GEMM dispatch of crates/prelude-cuda/src/ops/gemm.rs:35-137 (library kernels there).
#include "block_core.h"
#include "api.h"

namespace pa {

enum BlockEpilogue : int { kBlockPlain = 0, kBlockGated = 1, kBlockSlices = 2 };
// What a kBlockGated epilogue makes of a lane's four sums (the launcher's `epilogue` less one).
enum BlockAct : int { kBlockSilu = 0, kBlockGelu = 1, kBlockClamped = 2, kBlockRelu2 = 3 };

struct BlockProduct {
  const bf16 *x, *w;
  const float* bias;
  void* c;
  int m, n, k;
  long ldx, ldc;
  int act;
  float limit, alpha;
};

template <typename Core, int COLS>
__device__ __forceinline__ void store_block(const BlockProduct& p, const bf16* out, int m0, int from, int left) {
  typedef BlockOut<Core, bf16, COLS> Out;
  __syncthreads();
  const int rows = p.m - m0 < Core::kRows ? p.m - m0 : Core::kRows;
  bf16* c = (bf16*)p.c + (size_t)m0 * p.ldc + from;
  if (p.ldc % 8 == 0) store_rows<bf16, COLS, Out::kPitch, 8>(c, p.ldc, out, rows, left);
  else store_rows<bf16, COLS, Out::kPitch, 2>(c, p.ldc, out, rows, left);   // rows that are not 16-byte aligned
}

// One workgroup's outputs: rows m0 .., columns n0 .., `steps` steps of 64 columns of K from s_begin.
template <typename Core, int EPI>
__device__ __forceinline__ void block_tile(const BlockProduct& p, unsigned char* lds_raw, int m0, int n0, int s_begin, int steps, int slice) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, g = lane / 16, r = lane % 16;
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_raw;
  const int steps_all = p.k / 64, tiles = p.n / 16;
  const bf16* x[Core::kLoadsX];
#pragma unroll
  for (int j = 0; j < Core::kLoadsX; ++j) {
    const int row = m0 + j * 64 + (int)threadIdx.x / 8;              // a row that does not exist: the last one, not stored
    x[j] = p.x + (size_t)(row < p.m ? row : p.m - 1) * p.ldx + s_begin * 64 + block_x_column(threadIdx.x);
  }
  const bf16* w[Core::kLoadsW];
#pragma unroll
  for (int j = 0; j < Core::kLoadsW; ++j) {
    const int t = n0 / 16 + j * 4 + wave / 2;
    w[j] = p.w + ((size_t)(t < tiles ? t : tiles - 1) * steps_all + s_begin) * 1024 + (wave % 2) * 512 + lane * 8;
  }
  f32x4 acc[Core::MT][Core::NT];
  Core::run(lds, x, w, steps, acc);

  // lane (g, r) holds four consecutive columns of row r of a tile
  __syncthreads();                                                   // everyone's loads have come, the operands have been read
  if constexpr (EPI == kBlockSlices) {
    typedef BlockOut<Core, float, Core::kCols> Out;
    float* out = reinterpret_cast<float*>(lds_raw);
    float* c = (float*)p.c + (size_t)slice * p.m * p.n + n0;
    const bool biased = p.bias && slice == 0;
#pragma unroll
    for (int t0 = 0; t0 < Core::MT; t0 += Core::kTiles0) {
      constexpr int kRows0 = Core::kRows0;
      if (t0) __syncthreads();
#pragma unroll
      for (int t = t0; t < Core::MT && t < t0 + Core::kTiles0; ++t)
#pragma unroll
        for (int u = 0; u < Core::NT; ++u) {
          const int row = Core::row_of(wave, t) + r - (t0 ? kRows0 : 0), col = Core::col_of(wave, u) + 4 * g;
          f32x4 v = acc[t][u];
          if (biased && n0 + col < p.n) v += *reinterpret_cast<const f32x4*>(p.bias + n0 + col);
          *reinterpret_cast<f32x4*>(out + row * Out::kPitch + col) = v;
        }
      __syncthreads();
      const int first = m0 + (t0 ? kRows0 : 0), most = t0 ? Core::kRows - kRows0 : kRows0;
      if (first < p.m)
        store_rows<float, Core::kCols, Out::kPitch, 4>(c + (size_t)first * p.n, p.n, out, p.m - first < most ? p.m - first : most, p.n - n0);
    }
  } else {
    bf16* out = reinterpret_cast<bf16*>(lds_raw);
    auto put = [&](auto of) {
#pragma unroll
      for (int t = 0; t < Core::MT; ++t)
#pragma unroll
        for (int u = 0; u < Core::NT; ++u) of(Core::row_of(wave, t) + r, Core::col_of(wave, u) + 4 * g, acc[t][u]);
    };
    auto pairs = [&](auto of) {
      put([&](int row, int col, const f32x4& v) {
        *reinterpret_cast<bf16x2*>(out + row * BlockOut<Core, bf16, Core::kCols / 2>::kPitch + col / 2) = bf16x2{(bf16)of(v[0], v[1]), (bf16)of(v[2], v[3])};
      });
    };
    auto each = [&](auto of) {
      put([&](int row, int col, const f32x4& v) {
        const f32x4 o = of(v, col);
        *reinterpret_cast<bf16x4*>(out + row * BlockOut<Core, bf16, Core::kCols>::kPitch + col) = bf16x4{(bf16)o[0], (bf16)o[1], (bf16)o[2], (bf16)o[3]};
      });
    };
    if (EPI == kBlockPlain) {
      if (p.bias) each([&](f32x4 v, int col) { return n0 + col < p.n ? v + *reinterpret_cast<const f32x4*>(p.bias + n0 + col) : v; });
      else each([](f32x4 v, int) { return v; });
      store_block<Core, Core::kCols>(p, out, m0, n0, p.n - n0);
    } else if (p.act == kBlockRelu2) {
      each([](f32x4 v, int) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = fmaxf(v[i], 0.f);
          v[i] *= v[i];
        }
        return v;
      });
      store_block<Core, Core::kCols>(p, out, m0, n0, p.n - n0);
    } else {
      if (p.act == kBlockSilu) pairs([](float gate, float up) { return gate_activation_of<bf16>(gate, kActSilu) * up; });
      else if (p.act == kBlockGelu) pairs([](float gate, float up) { return gate_activation_of<bf16>(gate, kActGeluTanh) * up; });
      else
        pairs([&](float gate, float up) {
          const float gc = fminf(gate, p.limit), uc = fminf(fmaxf(up, -p.limit), p.limit);
          return gc * sigmoid_of<bf16>(p.alpha * gc) * (uc + 1.0f);
        });
      store_block<Core, Core::kCols / 2>(p, out, m0, n0 / 2, (p.n - n0) / 2);
    }
  }
}

// The tiles of one slice are numbered by groups of `group` row tiles, the row tiles of a column tile side by side; with HALF,
// those from `whole` on are two workgroups each, of half the columns: what is left after whole rounds of the chip then takes
// little more than half a round.
template <typename Core, typename Half, int EPI>
__global__ __launch_bounds__(kBlockThreads, 2) void gemm_block_kernel(BlockProduct p, int row_tiles, int col_tiles, int group, int sps,
                                                                      int whole) {
  constexpr bool kHalves = !__is_same(Half, void);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  int id, half = -1;
  if (!kHalves || (int)blockIdx.x < whole) {
    id = block_place(blockIdx.x, kHalves ? whole : (int)gridDim.x);
  } else {
    const int h = block_place(blockIdx.x - whole, gridDim.x - whole);
    id = whole + h / 2;
    half = h % 2;
  }
  const int tiles = row_tiles * col_tiles, slice = id / tiles;
  id -= slice * tiles;
  const int first = id / (group * col_tiles) * group, within = id % (group * col_tiles);
  const int rows = row_tiles - first < group ? row_tiles - first : group;
  const int m0 = (first + within % rows) * Core::kRows, n0 = within / rows * Core::kCols;
  const int steps_all = p.k / 64, s_begin = slice * sps;
  const int steps = s_begin + sps < steps_all ? sps : steps_all - s_begin;
  if constexpr (kHalves) {
    if (half >= 0) {
      const int nh = n0 + half * Half::kCols;
      if (nh < p.n) block_tile<Half, EPI>(p, lds_raw, m0, nh, s_begin, steps, slice);
      return;
    }
  }
  block_tile<Core, EPI>(p, lds_raw, m0, n0, s_begin, steps, slice);
}

// The shapes, and what was measured of them: us a step of 64 columns with every compute unit at work (weights of 2,560 x 9,728,
// 6,144 x 2,560 and 4,096, 4,096 x 1,024 by 128 to 2,048 rows inside graphs), and what a round takes besides of a product left whole: each
// of 256 x 256 (weights of 8,192 rows and 1,024 to 3,584 columns by 2,048 rows take 6 to 8 us more than the steps say, half a round of
// halves 3 to 6; from 2.5 on the line against the library comes right: of 473 products 35 more than 3 % behind it for 2.5, 34 for 5, 50 for
// none) and each behind the first of 64 x 128 ([19456, 2560] by 160 rows 41 us where the steps say 36.6, in one round of 192 x 128 37).
// All of this is from before the outputs left through LDS (2 to 4 us less a round) and the last two went in step (some 0.05 less a
// step): the numbers are an order of choice by now and no longer times, see block_price for what the choice costs.
struct BlockShape {
  int rows, cols;
  double step, whole, next;
};
constexpr BlockShape kBlockShapes[] = {
    {256, 256, 1.33, 2.5, 0.}, {256, 192, 1.18, 0., 0.}, {192, 256, 1.15, 0., 0.}, {192, 192, 0.98, 0., 0.}, {256, 128, 0.82, 0., 0.},
    {192, 128, 0.70, 0., 0.},  {128, 128, 0.58, 0., 0.}, {64, 128, 0.32, 0., 2.0}, {64, 64, 0.22, 0., 0.},
};
constexpr int kBlockShapeCount = sizeof(kBlockShapes) / sizeof(kBlockShapes[0]);

inline long block_whole(long tiles) {                                // see gemm_block_kernel: tiles that are not halved
  const long rest = tiles % 256;
  return rest > 128 ? tiles : tiles - rest;
}

// What a product takes as `shape` and `slices`, in us: a launch, and for every round of the chip its steps and what the first
// loads and the stores take; slices are written and read again as 32-bit numbers.  Over the 24 weights of a layer of models of 0.6B to
// 32B by 65 to 2,048 rows, with the reader of slices behind them, the shape so priced least takes more than a twentieth longer than the
// fastest in two of 216 products if the number of slices is left as it is, and the two together in 23, in nine more than a tenth, a fifth
// at most: the slices of narrow weights, too few of them ([5120, 25600] by 96 rows 70.2 us in three, 58.1 in six of 128 x 128).
inline double block_price(int shape, int slices, int m, int n, int k) {
  const BlockShape& s = kBlockShapes[shape];
  const int steps = k / 64, sps = (steps + slices - 1) / slices;
  const long tiles = (long)((m + s.rows - 1) / s.rows) * ((n + s.cols - 1) / s.cols);
  const double round = 2.0 + (s.rows * s.cols >= 192 * 128 ? 1.5 : 0.0) + sps * s.step + (slices == 1 ? s.whole : 0.0);
  double rounds;
  if (shape == 0 && slices == 1) {
    const long whole = block_whole(tiles);
    rounds = (double)((whole + 255) / 256) + (whole < tiles ? 0.62 : 0.0);
  } else {
    rounds = (double)((tiles * slices + 255) / 256);
  }
  const double extra = slices > 1 ? (double)m * n * (8.0 * slices - 4.0) / 5.5e6 : 0.0;
  const double weight = 2.0 * n * k;                                 // from memory, once: at 4.6 TB/s where nothing else takes as long
  const double next = slices == 1 && rounds > 1.0 ? (rounds - 1.0) * s.next : 0.0;
  const double time = 2.0 + rounds * round + next + weight / 2e7;
  return (time > 5.5 + weight / 4.6e6 ? time : 5.5 + weight / 4.6e6) + extra;
}

template <typename Core, typename Half, int EPI>
int launch_block(hipStream_t st, const BlockProduct& p, int slices) {
  auto* kernel = &gemm_block_kernel<Core, Half, EPI>;
  constexpr size_t kOut = EPI == kBlockSlices ? BlockOut<Core, float, Core::kCols>::kBytes : BlockOut<Core, bf16, Core::kCols>::kBytes;
  constexpr size_t kLds = kOut > Core::kLds ? kOut : Core::kLds;
  static_assert(kLds <= 160 * 1024, "a compute unit's LDS");
  // more LDS than a kernel may declare: asked for at launch, allowed once per kernel
  static const hipError_t allowed =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
  if (allowed != hipSuccess) return pa::fail("gemm_block: %zu bytes of LDS refused: %s", kLds, hipGetErrorString(allowed));
  const int row_tiles = (p.m + Core::kRows - 1) / Core::kRows, col_tiles = (p.n + Core::kCols - 1) / Core::kCols;
  const int steps = p.k / 64, sps = (steps + slices - 1) / slices;
  const long tiles = (long)row_tiles * col_tiles;
  const long whole = __is_same(Half, void) ? tiles * slices : block_whole(tiles);
  const long blocks = __is_same(Half, void) ? whole : whole + 2 * (tiles - whole);
  PA_REQUIRE(blocks < (1L << 31), "gemm_block: %ld workgroups", blocks);
  // eight row tiles of 256 rows side by side (2,048 rows of X: an L2 holds a step of them many times over)
  const int group = 2048 / Core::kRows;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kBlockThreads), kLds, st, p, row_tiles, col_tiles, group, sps, (int)whole);
  return check_launch("gemm_block");
}

template <int EPI>
int launch_block_shape(hipStream_t st, const BlockProduct& p, int slices, int shape) {
  switch (shape) {
    case 0:
      if constexpr (EPI == kBlockSlices) return launch_block<BlockTwoPhase<4, 4, 2, 2, 4>, void, EPI>(st, p, slices);
      else return launch_block<BlockTwoPhase<4, 4, 2, 2, 4>, BlockTwoPhase<4, 4, 1, 1, 4>, EPI>(st, p, slices);
    case 1: return launch_block<BlockTwoPhase<4, 4, 2, 1, 4>, void, EPI>(st, p, slices);
    case 2: return launch_block<BlockTwoPhase<4, 2, 2, 2, 4>, void, EPI>(st, p, slices);
    case 3: return launch_block<BlockTwoPhase<4, 2, 2, 1, 4>, void, EPI>(st, p, slices);
    case 4: return launch_block<BlockOnePhase<4, 2, 4, 4, 1, 3>, void, EPI>(st, p, slices);
    case 5: return launch_block<BlockOnePhase<4, 2, 3, 4, 1, 4>, void, EPI>(st, p, slices);
    case 6: return launch_block<BlockOnePhase<2, 4, 4, 2, 1, 5>, void, EPI>(st, p, slices);
    case 7: return launch_block<BlockInStep<2, 4, 2, 2, 2, 3>, void, EPI>(st, p, slices);
    case 8: return launch_block<BlockInStep<2, 4, 2, 1, 2, 4>, void, EPI>(st, p, slices);
  }
  return pa::fail("gemm_block: no shape %d", shape);
}

}  // namespace pa

using namespace pa;

// The shape and the number of slices (least to most, more than one only of four steps or more each) that are priced least for
// a product of m rows by an [n, k] weight: out[0], out[1]; the price in us in `price`.
extern "C" void pa_gemm_block_plan(int m, int n, int k, int least, int most, int* out, double* price) {
  const int steps = k / 64;
  out[0] = 0, out[1] = least;
  double best = -1.0;
  for (int slices = least; slices <= most; ++slices) {
    if (slices > least && steps / slices < 4) break;
    const int sps = (steps + slices - 1) / slices;
    if ((steps + sps - 1) / sps != slices) continue;
    for (int shape = 0; shape < kBlockShapeCount; ++shape) {
      const double p = block_price(shape, slices, m, n, k);
      if (best < 0.0 || p < best) best = p, out[0] = shape, out[1] = slices;
    }
  }
  *price = best;
}

// C[m, n] = X[m, k] W^T from the weight in tiles, any m, n a multiple of 16, k of 64.  slices 1: epilogue 0 writes C (+ bias) in
// bfloat16, 1 and 2 C[m, n/2] = SiLU or GELU-tanh(gate) * up, 3 the clamped gated pair, 4 the square of relu.  slices > 1
// (epilogue 0 alone): C [slices, m, n] receives each slice's 32-bit sums (the bias in the first).  shape: an index into
// kBlockShapes; the sums of a slice are the same bits at every shape.
extern "C" int pa_gemm_block(void* stream, int epilogue, const void* x, const void* w, const float* bias, void* c, int m, int n, int k,
                             long ldx, long ldc, int slices, int shape, float limit, float alpha) {
  if (m == 0 || n == 0) return 0;
  PA_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_block: bad sizes m=%d n=%d k=%d", m, n, k);
  PA_REQUIRE(n % 16 == 0 && k % 64 == 0, "gemm_block: n=%d must be a multiple of 16 and k=%d of 64", n, k);
  PA_REQUIRE(ldx >= k && ldx % 8 == 0, "gemm_block: the row stride %ld must be a multiple of 8 and at least k=%d", ldx, k);
  PA_REQUIRE(x && w && c, "gemm_block: an operand is missing");
  PA_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)c) % 16 == 0 && (uintptr_t)bias % 16 == 0, "gemm_block: operands must be 16-byte aligned");
  const int steps = k / 64;
  PA_REQUIRE(slices >= 1 && slices <= steps, "gemm_block: %d slices of %d steps", slices, steps);
  {
    const int sps = (steps + slices - 1) / slices;   // every slice must get a step, or its part would stay unwritten
    PA_REQUIRE((steps + sps - 1) / sps == slices, "gemm_block: %d steps do not cut into %d slices of %d", steps, slices, sps);
  }
  PA_REQUIRE(epilogue >= 0 && epilogue <= 1 + kBlockRelu2, "gemm_block: unknown epilogue %d", epilogue);
  const bool pairs = epilogue >= 1 && epilogue <= 1 + kBlockClamped;
  PA_REQUIRE(epilogue == 0 || (!bias && slices == 1), "gemm_block: an activation needs whole sums and no bias");
  PA_REQUIRE(epilogue != 1 + kBlockClamped || limit > 0.f, "gemm_block: clamped gated pairs need a clamp > 0, not %g", (double)limit);
  PA_REQUIRE(slices > 1 || (ldc >= (pairs ? n / 2 : n) && ldc % (pairs ? 2 : 4) == 0), "gemm_block: bad output row stride %ld", ldc);
  hipStream_t st = (hipStream_t)stream;
  const BlockProduct p{(const bf16*)x, (const bf16*)w, bias, c, m, n, k, ldx, ldc, epilogue - 1, limit, alpha};
  if (slices > 1) return launch_block_shape<kBlockSlices>(st, p, slices, shape);
  if (epilogue == 0) return launch_block_shape<kBlockPlain>(st, p, 1, shape);
  return launch_block_shape<kBlockGated>(st, p, 1, shape);
}
