// Products with a weight per group of rows, on the matrix cores (bfloat16, 32-bit sums): the experts' products
// (group = expert, rows = the step's entries in expert order) and the per-head maps of attention through a latent
// (group = head, rows = tokens).
//
// y[row, n] = sum_k x[row, k] * w[group, n, k], every group's weight in tiles of 16 outputs x 64 columns in the order a
// wavefront's lanes load them (pa_pack_tiles; outputs and columns that do not exist are zeros): a load of a fragment is
// 1 KB of consecutive memory, where rows as stored gave sixteen half lines.  W^T tile as A (row = output), X^T as B
// (column = row of x), v_mfma_f32_16x16x32_bf16: lane (g, r) of a step holds columns 16 g .. 16 g + 15 of row r on both
// sides, the first eight for one product and the others for the next, and ends with outputs 4g..4g+3 of row r of x.
#include "block_core.h"
#include "api.h"

#include <type_traits>

namespace pa {

struct GroupFrag {
  bf16x8 lo, hi;
};

__device__ __forceinline__ GroupFrag group_load_w(const bf16* tile, int step, int lane) {
  GroupFrag f;
  const bf16* p = tile + (size_t)step * 1024 + lane * 8;
  f.lo = *reinterpret_cast<const bf16x8*>(p);
  f.hi = *reinterpret_cast<const bf16x8*>(p + 512);
  return f;
}

// Columns at .. at + 15 of a row of x; a half past the row's end (K is a multiple of 8) reads the row's first columns, which
// are taken out again (group_cut) where they would be multiplied: an infinity among them times a zero of the tile is NaN.
__device__ __forceinline__ GroupFrag group_load_x(const bf16* row, int at, int K) {
  GroupFrag f;
  f.lo = *reinterpret_cast<const bf16x8*>(row + (at + 8 <= K ? at : 0));
  f.hi = *reinterpret_cast<const bf16x8*>(row + (at + 16 <= K ? at + 8 : 0));
  return f;
}

__device__ __forceinline__ void group_cut(GroupFrag& f, int at, int K) {
  f.lo = at + 8 <= K ? f.lo : bf16x8{};
  f.hi = at + 16 <= K ? f.hi : bf16x8{};
}

// A lane's four outputs nb .. nb + 3 of one row: act 0 as they are, 1 the square of relu, 2 clamped and 3 plain gated
// pairs (gate, up), one output a pair and rows of N / 2; in one store where `whole` says that rows are aligned whole
// fours, or pairs of gated outputs (a store an output cost the many-row product a quarter of its time).
template <typename TY>
__device__ __forceinline__ void group_store(TY* __restrict__ y, const f32x4 v, int nb, int N, bool whole, int act, float limit, float alpha) {
  typedef TY y2 __attribute__((ext_vector_type(2)));
  typedef TY y4 __attribute__((ext_vector_type(4)));
  if (act >= 2) {
    float o[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      o[i] = act == 2 ? clamped_gate(v[2 * i], v[2 * i + 1], limit, alpha) : gate_activation(v[2 * i], kActSilu) * v[2 * i + 1];
    if (whole && nb + 3 < N) {
      *reinterpret_cast<y2*>(y + nb / 2) = y2{from_f32<TY>(o[0]), from_f32<TY>(o[1])};
      return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (nb + 2 * i < N) y[nb / 2 + i] = from_f32<TY>(o[i]);
    return;
  }
  f32x4 u = v;
  if (act == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u[i] = fmaxf(u[i], 0.f);
      u[i] = u[i] * u[i];
    }
  }
  if (whole && nb + 3 < N) {
    *reinterpret_cast<y4*>(y + nb) = y4{from_f32<TY>(u[0]), from_f32<TY>(u[1]), from_f32<TY>(u[2]), from_f32<TY>(u[3])};
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (nb + i < N) y[nb + i] = from_f32<TY>(u[i]);
}

// Heads, and one weight for a few rows: what counts is how fast the weights stream, so a workgroup owns no more than NT tiles
// of 16 outputs of one group (and 16 RM rows), its wavefronts take the steps of k in turn, one step in flight while one is
// multiplied, and are summed through LDS in their order.  (The experts' products, which have tiles enough for a wavefront
// each, are moe_few_mfma_kernel's.)
// xrow(m) / yrow(m): element offsets of row m's input and output.
template <typename TY, int RM, int NT, int WAVES, typename RowX, typename RowY>
__device__ __forceinline__ void group_few(const bf16* __restrict__ x, const bf16* __restrict__ w, TY* __restrict__ y, int K, int N,
                                          int n_rows, int tile0, bool whole, int act, float limit, float alpha, RowX xrow, RowY yrow) {
  static_assert(NT * RM <= WAVES, "a wavefront finishes one tile");
  __shared__ __attribute__((aligned(16))) float red[WAVES][NT * RM][kWave][4];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int steps = (K + 63) / 64, tiles = (N + 15) / 16;
  const bf16* wt[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) wt[u] = w + (size_t)(tile0 + u < tiles ? tile0 + u : tiles - 1) * steps * 1024;
  const bf16* xr[RM];
#pragma unroll
  for (int t = 0; t < RM; ++t) xr[t] = x + xrow(16 * t + r < n_rows ? 16 * t + r : 0);   // rows that do not exist: one that does, not stored
  f32x4 acc[NT][RM];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < RM; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  GroupFrag wn[NT], xn[RM];
  auto load = [&](int s) {                                       // no load under a condition: past the end the last step, not multiplied
    s = s < steps ? s : steps - 1;
#pragma unroll
    for (int u = 0; u < NT; ++u) wn[u] = group_load_w(wt[u], s, lane);
#pragma unroll
    for (int t = 0; t < RM; ++t) xn[t] = group_load_x(xr[t], s * 64 + 16 * g, K);
  };
  auto walk = [&](auto ragged) {
    load(wave);
    for (int s = wave; s < steps; s += WAVES) {
      GroupFrag wc[NT], xc[RM];
#pragma unroll
      for (int u = 0; u < NT; ++u) wc[u] = wn[u];
#pragma unroll
      for (int t = 0; t < RM; ++t) xc[t] = xn[t];
      load(s + WAVES);
      if constexpr (decltype(ragged)::value) {                   // a select, not a branch: the loads stay ahead
#pragma unroll
        for (int t = 0; t < RM; ++t) group_cut(xc[t], s * 64 + 16 * g, K);
      }
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int t = 0; t < RM; ++t) {
          acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[u].lo, xc[t].lo, acc[u][t], 0, 0, 0);
          acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[u].hi, xc[t].hi, acc[u][t], 0, 0, 0);
        }
    }
  };
  if (K % 64 == 0) walk(std::false_type());
  else walk(std::true_type());
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < RM; ++t) *reinterpret_cast<f32x4*>(red[wave][u * RM + t][lane]) = acc[u][t];
  __syncthreads();
  if (wave >= NT * RM) return;
  const int u = wave / RM, t = wave % RM;
  f32x4 v = *reinterpret_cast<const f32x4*>(red[0][wave][lane]);
#pragma unroll
  for (int q = 1; q < WAVES; ++q) v += *reinterpret_cast<const f32x4*>(red[q][wave][lane]);
  if (16 * t + r >= n_rows) return;
  group_store(y + yrow(16 * t + r), v, 16 * (tile0 + u) + 4 * g, N, whole, act, limit, alpha);
}

// Which expert a work item belongs to.  An expert with c entries has ceil(c / rows) tiles of positions, each against
// `chunks` chunks of outputs; the items are numbered expert by expert, chunk by chunk, the tiles of one chunk side by
// side.  The launch is a line of workgroups that the hardware deals out to the eight XCDs in turn (each with an L2 of
// its own), and every XCD is given one stretch of the items that there are: an expert's rows and a chunk of its weight
// then stay in one L2 while its tiles need them.  An expert's entries are shared out evenly over its tiles, in whole
// sixteens.  False for a workgroup beyond the last item.  All lanes of a wavefront call it with the same arguments;
// every lane takes an expert (64 at a time), so that no chain of dependent loads runs over the experts.
struct GroupItem {
  int e, p0, rows, chunk;
};

// The running total over a wavefront's lanes, each with its own in it, by the vector ALU's exchanges: within rows of sixteen, then
// the rows' totals to the rows behind.
__device__ __forceinline__ int running_total(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into the odd rows
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into the upper half
  return v;
}

__device__ __forceinline__ bool find_item(const int* __restrict__ offsets, int experts, int rows, int chunks, GroupItem& out) {
  const int lane = threadIdx.x % kWave;
  // the lane's expert of those from `base` on: its first entry and the one behind its last
  auto entries = [&](int base, int& a, int& b) {
    const int e = base + lane;
    a = offsets[e < experts ? e : experts];
    b = offsets[e < experts ? e + 1 : experts];
  };
  int a, b, total = 0;
  for (int base = 0; base < experts; base += kWave) {
    entries(base, a, b);
    total += __builtin_amdgcn_readlane(running_total((b - a + rows - 1) / rows), kWave - 1);
  }
  total *= chunks;
  const int per_xcd = (total + 7) / 8;
  const int at = (int)(blockIdx.x / 8), item = (int)(blockIdx.x % 8) * per_xcd + at;
  if (at >= per_xcd || item >= total) return false;
  const int tile = item / chunks;
  int before = 0;                                              // tiles of the experts of earlier rounds
  for (int base = 0; base < experts; base += kWave) {
    if (experts > kWave) entries(base, a, b);
    const int mine = (b - a + rows - 1) / rows, incl = running_total(mine);
    const unsigned long long hit = __ballot(before + incl > tile);
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      const int n = __builtin_amdgcn_readlane(mine, src);
      const int within = item - (before + __builtin_amdgcn_readlane(incl, src) - n) * chunks;
      const int ea = __builtin_amdgcn_readlane(a, src), c = __builtin_amdgcn_readlane(b, src) - ea;
      const int share = (c + 16 * n - 1) / (16 * n) * 16;      // rows a tile, no more than `rows` (a multiple of 16)
      const int p = within % n * share;
      out.e = base + src;
      out.chunk = within / n;
      out.p0 = ea + p;
      out.rows = c - p < share ? c - p : share;
      return out.rows > 0;                                     // (sixteens can leave the last tile without a row)
    }
    before += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  return false;
}

// The experts' product for few rows: a workgroup is one wavefront with NT tiles of 16 outputs of one expert and 16 RM of its
// positions, and walks k in order, D steps in flight; a step is multiplied before the step D further on is asked for in its
// registers.  A sum is then one chain over k, as in the kernel for many rows below: a position's outputs are the same bits
// whichever kernel the step's size takes.  What bounds it is how fast the weights stream: 48 entries over 64 experts of
// [1408, 2048] read some 196 MB in 37.2 us, of [2048, 1408] in 39.6 (38.0 and 39.3 with eight wavefronts a tile that
// shared k, whose sums were others than the many rows'), 510 entries 61.4 and 67.0 (66.5 and 71.5), 768 with 32 positions
// 65.0 and 69.5 (68.1 and 74.1); 96 are the one size measured that lost, 50.1 and 56.2 (50.0 and 52.3).  One wavefront a
// tile is enough for that because 12 a compute unit fit and each has 16 KB on its way.
// `from_tokens`: position p reads row order[p] / top of x.
template <typename TY, int RM, int NT, int D>
__global__ __launch_bounds__(kWave) void moe_few_mfma_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, TY* __restrict__ y,
                                                             const int* __restrict__ offsets, const int* __restrict__ order,
                                                             int experts, int top, int K, int N, int chunks, int from_tokens, bool whole,
                                                             int act, float limit, float alpha) {
  GroupItem it;
  if (!find_item(offsets, experts, 16 * RM, chunks, it)) return;
  const int lane = threadIdx.x, g = lane / 16, r = lane % 16;
  const int steps = (K + 63) / 64, tiles = (N + 15) / 16, last = steps - 1, tile0 = it.chunk * NT;
  const bf16* we = w + (size_t)it.e * tiles * steps * 1024;
  const bf16* wt[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) wt[u] = we + (size_t)(tile0 + u < tiles ? tile0 + u : tiles - 1) * steps * 1024;
  const bf16* xr[RM];
#pragma unroll
  for (int t = 0; t < RM; ++t) {
    const int p = it.p0 + (16 * t + r < it.rows ? 16 * t + r : 0);   // rows that do not exist: one that does, not stored
    xr[t] = x + (size_t)(from_tokens ? order[p] / top : p) * K;
  }
  f32x4 acc[NT][RM];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < RM; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  GroupFrag wf[D][NT], xf[D][RM];
  auto load = [&](int d, int s) {                                // no load under a condition: past the end the last step, not multiplied
    s = s < steps ? s : last;
#pragma unroll
    for (int u = 0; u < NT; ++u) wf[d][u] = group_load_w(wt[u], s, lane);
#pragma unroll
    for (int t = 0; t < RM; ++t) xf[d][t] = group_load_x(xr[t], s * 64 + 16 * g, K);
  };
  auto multiply = [&](int d) {
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int t = 0; t < RM; ++t) {
        acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[d][u].lo, xf[d][t].lo, acc[u][t], 0, 0, 0);
        acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[d][u].hi, xf[d][t].hi, acc[u][t], 0, 0, 0);
      }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  int s0 = 0;
  for (; s0 + D < steps; s0 += D)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      multiply(d);
      load(d, s0 + d + D);
    }
#pragma unroll
  for (int d = 0; d < D; ++d) {                                  // the last one to D steps
    const int s = s0 + d;
    if (s >= steps) continue;
    if (s == last)
#pragma unroll
      for (int t = 0; t < RM; ++t) group_cut(xf[d][t], s * 64 + 16 * g, K);
    multiply(d);
  }
#pragma unroll
  for (int t = 0; t < RM; ++t) {
    if (16 * t + r >= it.rows) continue;
    TY* yr = y + (size_t)(it.p0 + 16 * t + r) * (act >= 2 ? N / 2 : N);
#pragma unroll
    for (int u = 0; u < NT; ++u)
      if (tile0 + u < tiles) group_store(yr, acc[u][t], 16 * (tile0 + u) + 4 * g, N, whole, act, limit, alpha);
  }
}

// The experts' product for many rows: a workgroup owns up to 128 positions of one expert and 192 outputs, a wavefront all
// of the positions and three tiles of outputs.  The rows of x go through LDS, 64 columns at a time, held in registers as
// many steps ahead of their use as the weight, which comes straight from memory; two buffers, rows of 160 bytes (16-byte
// reads of sixteen rows at full rate).  Everything is asked for the same two steps ahead, no load under a condition, so
// that a wait is for no more than it must be (four steps ahead are no faster).  Tiles of rows that do not exist cost no products.
// 12,288 entries over 64 experts of [1408, 2048] take 116 us (211 with steps of 32 columns, one ahead, weights as
// stored), of [2048, 1408] 137 (229).
constexpr int kGbTiles = 8, kGbRows = 16 * kGbTiles, kGbCols = 3, kGbDepth = 2;
constexpr int kGbStride = 64 + 16;   // elements of an LDS row

template <typename TY>
__global__ __launch_bounds__(256, 2) void moe_many_mfma_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, TY* __restrict__ y,
                                                               const int* __restrict__ offsets, const int* __restrict__ order,
                                                               int experts, int top, int K, int N, int chunks, int from_tokens,
                                                               bool whole, int act, float limit, float alpha) {
  constexpr int MT = kGbTiles, NT = kGbCols, D = kGbDepth, PIECES = kGbRows * 8 / 256;
  __shared__ __attribute__((aligned(16))) bf16 xs[2][kGbRows][kGbStride];
  GroupItem it;
  if (!find_item(offsets, experts, kGbRows, chunks, it)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int steps = (K + 63) / 64, tiles = (N + 15) / 16, last = steps - 1;
  const int n_rows = __builtin_amdgcn_readfirstlane(it.rows), tile0 = (it.chunk * 4 + wave) * NT;
  const bf16* we = w + (size_t)it.e * tiles * steps * 1024;
  const bf16* wt[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wt[j] = we + (size_t)(tile0 + j < tiles ? tile0 + j : tiles - 1) * steps * 1024;
  // piece p = thread + 256 j of a step: columns 8 (p % 8) .. of row p / 8
  const int col = 8 * (threadIdx.x % 8);
  const bf16* src[PIECES];
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int m = (threadIdx.x + 256 * j) / 8;
    const int p = it.p0 + (m < n_rows ? m : 0);
    src[j] = x + (size_t)(from_tokens ? order[p] / top : p) * K;
  }
  bf16x8 staged[D][PIECES];
  auto stage_load = [&](int set, int step) {
    const int at = (step < steps ? step : last) * 64 + col;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) staged[set][j] = *reinterpret_cast<const bf16x8*>(src[j] + (at + 8 <= K ? at : 0));
  };
  auto stage_store = [&](int set, int buf, int step) {
    if (step == last && last * 64 + col + 8 > K) {               // columns past the row's end: zeros
#pragma unroll
      for (int j = 0; j < PIECES; ++j) staged[set][j] = bf16x8{};
    }
#pragma unroll
    for (int j = 0; j < PIECES; ++j) *reinterpret_cast<bf16x8*>(&xs[buf][(threadIdx.x + 256 * j) / 8][col]) = staged[set][j];
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  GroupFrag wb[D][NT];
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int j = 0; j < NT; ++j) wb[d][j] = group_load_w(wt[j], d < steps ? d : last, lane);
#pragma unroll
  for (int d = 0; d < D; ++d) stage_load(d, d);
  stage_store(0, 0, 0);
  stage_load(0, D);
  __syncthreads();
  for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int s = s0 + u, buf = u & 1;
      GroupFrag wc[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) wc[j] = wb[u][j];
      stage_store((u + 1) % D, buf ^ 1, s + 1);                // (everyone left that buffer at the barrier before this step)
      stage_load((u + 1) % D, s + 1 + D);
#pragma unroll
      for (int j = 0; j < NT; ++j) wb[u][j] = group_load_w(wt[j], s + D < steps ? s + D : last, lane);
      if (s < steps) {
        GroupFrag xf[2];                                       // a row tile's fragments, read under the products of the one before
        auto fetch = [&](int t) {
          const bf16* at = &xs[buf][16 * t + r][16 * g];
          xf[t & 1].lo = *reinterpret_cast<const bf16x8*>(at);
          xf[t & 1].hi = *reinterpret_cast<const bf16x8*>(at + 8);
        };
        fetch(0);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          if (t + 1 < MT) fetch(t + 1);
          if (16 * t < n_rows) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
              acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[j].lo, xf[t & 1].lo, acc[t][j], 0, 0, 0);
              acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[j].hi, xf[t & 1].hi, acc[t][j], 0, 0, 0);
            }
          }
        }
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (16 * t + r >= n_rows) continue;
    TY* yr = y + (size_t)(it.p0 + 16 * t + r) * (act >= 2 ? N / 2 : N);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (tile0 + j < tiles) group_store(yr, acc[t][j], 16 * (tile0 + j) + 4 * g, N, whole, act, limit, alpha);
  }
}

// The experts' product for many rows, both operands through LDS (block_core.h): a workgroup owns up to 256 positions of one
// expert, in 128, 192 or 256 rows as it has positions, and COLS outputs.  The sums are those of the kernels above, bit for bit.
// 12,288 entries over 64 experts of [1408, 2048] take 94 us (moe_many_mfma_kernel 125), of [2048, 1408] 112 (140), where the weights
// alone, 369 MB, take 60 at the rate of a kernel that only reads: two rounds of the chip, each some 38 us of steps at 5 TB/s from memory
// and 8 before and behind them (10 before the item's search went by the vector ALU's exchanges and the outputs through LDS: 99 and 119);
// 8,400 entries 84 and 100 (121 and 126).  Up to 96 entries an expert that kernel takes no longer (6,000 entries 80 and 98).
constexpr int kMoeBlockRows = 256;
constexpr size_t kMoeBlockLds = 136 * 1024;                       // the ring, 128 KB, or the outputs behind it

template <typename Core, typename TY, bool PAIRS>
__device__ __forceinline__ void moe_block_item(const bf16* __restrict__ x, const bf16* __restrict__ w, TY* __restrict__ y,
                                               const int* __restrict__ order, int e, int p0, int n_rows, int n0, unsigned char* lds_raw,
                                               int top, int K, int N, int from_tokens, bool whole, bool aligned, int act, float limit,
                                               float alpha) {
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_raw;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, g = lane / 16, r = lane % 16;
  const int steps = K / 64, tiles = (N + 15) / 16;
  const bf16* xp[Core::kLoadsX];
#pragma unroll
  for (int j = 0; j < Core::kLoadsX; ++j) {
    const int m = j * 64 + (int)threadIdx.x / 8;
    const int p = p0 + (m < n_rows ? m : 0);                     // rows that do not exist: one that does, not stored
    xp[j] = x + (size_t)(from_tokens ? order[p] / top : p) * K + block_x_column(threadIdx.x);
  }
  const bf16* wp[Core::kLoadsW];
#pragma unroll
  for (int j = 0; j < Core::kLoadsW; ++j) {
    const int t = n0 / 16 + j * 4 + wave / 2;
    wp[j] = w + ((size_t)e * tiles + (t < tiles ? t : tiles - 1)) * steps * 1024 + (wave % 2) * 512 + lane * 8;
  }
  f32x4 acc[Core::MT][Core::NT];
  Core::run(lds, xp, wp, steps, acc);
  const int width = PAIRS ? N / 2 : N;
  if (aligned) {                                                 // through LDS, in whole rows
    constexpr int kCols = PAIRS ? Core::kCols / 2 : Core::kCols, kTiles0 = sizeof(TY) == 4 ? Core::kTiles0 : Core::MT;
    typedef BlockOut<Core, TY, kCols> Out;
    static_assert(Out::kBytes <= kMoeBlockLds, "what the launch asks for");
    TY* out = reinterpret_cast<TY*>(lds_raw);
    const int from = PAIRS ? n0 / 2 : n0;
    auto leave = [&](auto of) {
#pragma unroll
      for (int t0 = 0; t0 < Core::MT; t0 += kTiles0) {
        const int base = t0 ? Core::kRows0 : 0;
        __syncthreads();                                         // what lay there has come and has been read
#pragma unroll
        for (int t = t0; t < Core::MT && t < t0 + kTiles0; ++t)
#pragma unroll
          for (int u = 0; u < Core::NT; ++u) {
            const f32x4 v = acc[t][u];
            TY* at = out + (Core::row_of(wave, t) + r - base) * Out::kPitch + (Core::col_of(wave, u) + 4 * g) / (PAIRS ? 2 : 1);
            if constexpr (PAIRS) {
              typedef TY y2 __attribute__((ext_vector_type(2)));
              *reinterpret_cast<y2*>(at) = y2{from_f32<TY>(of(v[0], v[1])), from_f32<TY>(of(v[2], v[3]))};
            } else {
              typedef TY y4 __attribute__((ext_vector_type(4)));
              *reinterpret_cast<y4*>(at) = y4{from_f32<TY>(of(v[0])), from_f32<TY>(of(v[1])), from_f32<TY>(of(v[2])), from_f32<TY>(of(v[3]))};
            }
          }
        __syncthreads();
        const int end = t0 || kTiles0 == Core::MT ? Core::kRows : Core::kRows0, rows = (n_rows < end ? n_rows : end) - base;
        if (rows > 0) store_rows<TY, kCols, Out::kPitch, Out::kVec>(y + (size_t)(p0 + base) * width + from, width, out, rows, width - from);
      }
    };
    if constexpr (PAIRS) {
      if (act == 2) leave([&](float gate, float up) { return clamped_gate(gate, up, limit, alpha); });
      else leave([](float gate, float up) { return gate_activation(gate, kActSilu) * up; });
    } else {
      if (act == 1) leave([](float v) { return fmaxf(v, 0.f) * fmaxf(v, 0.f); });
      else leave([](float v) { return v; });
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < Core::MT; ++t) {
    const int m = Core::row_of(wave, t) + r;
    if (m >= n_rows) continue;
    TY* yr = y + (size_t)(p0 + m) * width;
#pragma unroll
    for (int u = 0; u < Core::NT; ++u) {
      const int n = n0 + Core::col_of(wave, u) + 4 * g;
      if (n < N) group_store(yr, acc[t][u], n, N, whole, PAIRS ? (act == 2 ? 2 : 3) : (act == 1 ? 1 : 0), limit, alpha);
    }
  }
}

// PAIRS: activations of gated pairs (act 2 and 3), else none or the square of relu.
template <typename TY, int COLS, bool PAIRS>
__global__ __launch_bounds__(kBlockThreads, 2) void moe_block_mfma_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                          TY* __restrict__ y, const int* __restrict__ offsets,
                                                                          const int* __restrict__ order, int experts, int top, int K, int N,
                                                                          int chunks, int from_tokens, bool whole, bool aligned, int act,
                                                                          float limit, float alpha) {
  constexpr int TN1 = COLS / 64 - 2;
  static_assert(COLS == 192 || COLS == 256, "two parts of outputs, the first 128");
  extern __shared__ __align__(16) unsigned char lds_raw[];
  GroupItem it;
  if (!find_item(offsets, experts, kMoeBlockRows, chunks, it)) return;
  const int e = __builtin_amdgcn_readfirstlane(it.e), p0 = __builtin_amdgcn_readfirstlane(it.p0);
  const int n_rows = __builtin_amdgcn_readfirstlane(it.rows), n0 = __builtin_amdgcn_readfirstlane(it.chunk) * COLS;
  auto item = [&](auto core) {
    using Core = decltype(core);
    static_assert(Core::kLds <= kMoeBlockLds && Core::kCols == COLS, "what the launch asks for");
    moe_block_item<Core, TY, PAIRS>(x, w, y, order, e, p0, n_rows, n0, lds_raw, top, K, N, from_tokens, whole, aligned, act, limit, alpha);
  };
  if (n_rows <= 128) item(BlockTwoPhase<2, 2, 2, TN1, 5>());
  else if (n_rows <= 192) item(BlockTwoPhase<4, 2, 2, TN1, 4>());
  else item(BlockTwoPhase<4, 4, 2, TN1, 4>());
}

// A part of every head's row beside its product, turned in pairs by the token's position (rotate_part): elements in_off .. of x
// to out_off .. of y.  In a launch of its own it took 4.1 us for 8 tokens, about what a launch costs; with the latents' norms
// split over two workgroups a decode step of 12 such layers went from 1,754 to 1,703 us.
struct HeadTurn {
  const float* inv_freq;
  const int* positions;
  int in_off, out_off, width, rot_dims;
};
constexpr int kTurnTokens = 16;   // a workgroup's

// Heads: grid (tiles of outputs within tiles of 16 RM tokens, then the parts that turn, heads); WAVES as many as there are steps of k, at most eight.
template <int RM, int NT, int WAVES>
__global__ __launch_bounds__(WAVES* kWave) void head_linear_mfma_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                        bf16* __restrict__ y, int tokens, int K, int N, long xs_t,
                                                                        long xs_h, long ys_t, long ys_h, bool whole, HeadTurn turn) {
  const int across = ((N + 15) / 16 + NT - 1) / NT, down = (tokens + 16 * RM - 1) / (16 * RM);
  if ((int)blockIdx.x >= across * down) {
    const int first = ((int)blockIdx.x - across * down) * kTurnTokens, items = turn.width - turn.rot_dims / 2;
    const int n = min(kTurnTokens, tokens - first) * items;
    for (int e = threadIdx.x; e < n; e += WAVES * kWave) {
      const int t = first + e / items;
      rotate_part(x + t * xs_t + blockIdx.y * xs_h + turn.in_off, y + t * ys_t + blockIdx.y * ys_h + turn.out_off, e % items,
                  (float)turn.positions[t], turn.inv_freq, turn.rot_dims);
    }
    return;
  }
  const int t0 = (int)(blockIdx.x / across) * 16 * RM, h = blockIdx.y;
  const int n_rows = tokens - t0 < 16 * RM ? tokens - t0 : 16 * RM;
  const size_t group = (size_t)((N + 15) / 16) * ((K + 63) / 64) * 1024;
  group_few<bf16, RM, NT, WAVES>(x, w + h * group, y, K, N, n_rows, (int)(blockIdx.x % across) * NT, whole, 0, 0.f, 0.f,
                                 [&](int m) { return (long)(t0 + m) * xs_t + (long)h * xs_h; },
                                 [&](int m) { return (long)(t0 + m) * ys_t + (long)h * ys_h; });
}

// One weight for a few rows with an activation on its outputs (act as above): what decode steps of a dense or shared
// feed-forward without a product of its own kind take, instead of a product and an elementwise launch behind it
// (bound by the weight's bytes or, small, by the launch: 8 rows of [1024, 2048] 3.7 us, 5.5 in two launches).
__global__ __launch_bounds__(512) void linear_few_mfma_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y,
                                                              int m, int K, int N, bool whole, int act, float limit, float alpha) {
  group_few<bf16, 1, 1, 8>(x, w, y, K, N, m, blockIdx.x, whole, act, limit, alpha, [&](int r) { return (long)r * K; },
                           [&](int r) { return (long)r * (act >= 2 ? N / 2 : N); });
}

}  // namespace pa

using namespace pa;

// Whether group_store may write a lane's outputs in one store: rows of y that start `stride` elements (of `size` bytes) apart.
static bool whole_stores(const void* y, size_t size, long stride, int act) {
  const int n = act >= 2 ? 2 : 4;
  return stride % n == 0 && (uintptr_t)y % (n * size) == 0;
}

constexpr long kMoeBlockMean = 96;   // below, the weights are what takes the time whichever kernel streams them

// Outputs a workgroup of moe_block_mfma_kernel takes: what leaves the chip the least idle, a round of it priced at its steps (as
// measured for products of that shape, gemm_block.hip) and what the first loads and the stores take.
static int moe_block_cols(long mean, int experts, int K, int N) {
  const long tiles = (mean + kMoeBlockRows - 1) / kMoeBlockRows * experts;
  const double step192 = mean <= 128 ? 0.7 : 1.1, step256 = mean <= 128 ? 0.78 : 1.25;
  const auto price = [&](int cols, double step) {
    return (double)((tiles * ((N + cols - 1) / cols) + 255) / 256) * (4.0 + K / 64 * step);
  };
  return price(192, step192) < price(256, step256) ? 192 : 256;
}

// x [rows, K] bfloat16 (a row per token when from_tokens, else per position), w [experts] of an [N, K] weight in tiles,
// y [entries, N] of y_dtype; K a multiple of 8.
extern "C" int pa_moe_linear_mfma(void* stream, int y_dtype, const void* x, const void* w, void* y, const int* offsets,
                                  const int* order, int entries, int experts, int top, int K, int N, int from_tokens, int act,
                                  float limit, float alpha) {
  if (entries == 0) return 0;
  PA_REQUIRE(entries > 0 && experts > 0 && top > 0 && K > 0 && N > 0 && K % 8 == 0, "moe_linear_mfma: bad sizes entries=%d experts=%d k=%d n=%d",
             entries, experts, K, N);
  PA_REQUIRE(act >= 0 && act <= 3, "moe_linear_mfma: unknown activation code %d", act);
  PA_REQUIRE(act < 2 || N % 2 == 0, "moe_linear_mfma: gated pairs need an even number of outputs");
  PA_REQUIRE(act != 2 || limit > 0.f, "moe_linear_mfma: clamped gated pairs need a clamp > 0");
  PA_REQUIRE(y_dtype == kBF16 || y_dtype == kF32, "moe_linear_mfma: unknown output type code %d", y_dtype);
  hipStream_t st = (hipStream_t)stream;
  // Entries an expert on average, and with them the rows a workgroup takes.  64 experts of [1408, 2048], us at 16 / 32 /
  // 128 rows: 61 / 65 / 66 with 8 entries an expert, 61 / 64 / 65 with 9, 81 / 66 / 67 with 18, 87 / 67 / 68 with 24, 96 / 77 / 69
  // with 30; of [2048, 1408]: 67 / 68 / 77, 68 / 68 / 78, 90 / 74 / 82, 95 / 77 / 83, 107 / 87 / 85.  The choice is one of speed
  // alone, every kernel gives the same bits.  It goes by the mean, for the host does not know how the entries fall: with all of
  // them on six experts 510 entries take 22 / 16 / 32 us and 1,536 (24 on average) 51 / 33 / 35.
  const long mean = entries / experts;
  const bool block = mean > kMoeBlockMean && K % 64 == 0 && ((uintptr_t)x & 15) == 0;
  const int cols = moe_block_cols(mean, experts, K, N);
  const int rows = block ? kMoeBlockRows : (mean <= 8 ? 16 : (mean <= 24 ? 32 : kGbRows));
  const int tiles = (N + 15) / 16, per_chunk = block ? cols / 16 : (rows == kGbRows ? 4 * kGbCols : (rows == 16 ? 2 : 4));
  const int chunks = (tiles + per_chunk - 1) / per_chunk;
  // no more tiles of positions than whole ones and one more for every expert that has entries
  const long most = entries / rows + (entries < experts ? entries : experts);
  const long items = most * chunks;
  PA_REQUIRE(items <= 0x7fffff00L, "moe_linear_mfma: %ld work items exceed the grid", items);
  const dim3 grid((unsigned)((items + 7) / 8 * 8));
  const bool whole = whole_stores(y, y_dtype == kBF16 ? sizeof(bf16) : sizeof(float), act >= 2 ? N / 2 : N, act);
  if (block) {
    const bool aligned = (act >= 2 ? N / 2 : N) * (y_dtype == kBF16 ? sizeof(bf16) : sizeof(float)) % 16 == 0 && (uintptr_t)y % 16 == 0;
    const auto launch = [&](auto* kernel, auto* out) {
      if (const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)kMoeBlockLds); e != hipSuccess)
        return pa::fail("moe_linear_mfma: %zu bytes of LDS refused: %s", kMoeBlockLds, hipGetErrorString(e));
      hipLaunchKernelGGL(kernel, grid, dim3(kBlockThreads), kMoeBlockLds, st, (const bf16*)x, (const bf16*)w, out, offsets, order, experts,
                         top, K, N, chunks, from_tokens, whole, aligned, act, limit, alpha);
      return check_launch("moe_linear_mfma");
    };
    const auto pick = [&](auto* out, auto pairs) {
      using TY = std::remove_pointer_t<decltype(out)>;
      constexpr bool kPairs = decltype(pairs)::value;
      return cols == 192 ? launch(&moe_block_mfma_kernel<TY, 192, kPairs>, out) : launch(&moe_block_mfma_kernel<TY, 256, kPairs>, out);
    };
    if (y_dtype == kBF16) return act >= 2 ? pick((bf16*)y, std::true_type()) : pick((bf16*)y, std::false_type());
    return act >= 2 ? pick((float*)y, std::true_type()) : pick((float*)y, std::false_type());
  }
#define PA_GM(KERNEL, THREADS)                                                                                              \
  do {                                                                                                                      \
    if (y_dtype == kBF16)                                                                                                   \
      hipLaunchKernelGGL((KERNEL(bf16)), grid, dim3(THREADS), 0, st, (const bf16*)x, (const bf16*)w, (bf16*)y, offsets,     \
                         order, experts, top, K, N, chunks, from_tokens, whole, act, limit, alpha);                                \
    else                                                                                                                    \
      hipLaunchKernelGGL((KERNEL(float)), grid, dim3(THREADS), 0, st, (const bf16*)x, (const bf16*)w, (float*)y, offsets,   \
                         order, experts, top, K, N, chunks, from_tokens, whole, act, limit, alpha);                                \
  } while (0)
#define PA_FEW16(TY) moe_few_mfma_kernel<TY, 1, 2, 4>
#define PA_FEW32(TY) moe_few_mfma_kernel<TY, 2, 4, 2>
#define PA_MANY(TY) moe_many_mfma_kernel<TY>
  if (rows == 16) PA_GM(PA_FEW16, kWave);
  else if (rows == 32) PA_GM(PA_FEW32, kWave);
  else PA_GM(PA_MANY, 256);
#undef PA_MANY
#undef PA_FEW32
#undef PA_FEW16
#undef PA_GM
  return check_launch("moe_linear_mfma");
}

// y[t, h, n] = sum_k x[t, h, k] w[h, n, k], w in tiles a head; strides in elements, x's multiples of 8 (16-byte pieces), y's
// any; K a multiple of 8.
extern "C" int pa_head_linear_mfma(void* stream, const void* x, const void* w, void* y, int tokens, int heads, int K, int N,
                                   long xs_t, long xs_h, long ys_t, long ys_h, const float* inv_freq, const int* positions,
                                   int in_off, int out_off, int width, int rot_dims) {
  if (tokens == 0) return 0;
  PA_REQUIRE(width >= 0 && rot_dims >= 0 && rot_dims <= width && rot_dims % 2 == 0 && (width == 0 || positions) && (rot_dims == 0 || inv_freq),
             "head_linear_mfma: a part of %d of which %d turn", width, rot_dims);
  PA_REQUIRE(width == 0 || (in_off >= 0 && out_off >= 0 && in_off + width <= xs_h && out_off + width <= ys_h),
             "head_linear_mfma: a part of %d at %d / %d does not fit heads of %ld / %ld", width, in_off, out_off, xs_h, ys_h);
  const HeadTurn turn{inv_freq, positions, in_off, out_off, width, rot_dims};
  const long turns = width ? (tokens + kTurnTokens - 1) / kTurnTokens : 0;
  PA_REQUIRE(tokens > 0 && heads > 0 && K > 0 && N > 0 && K % 8 == 0 && xs_t % 8 == 0 && xs_h % 8 == 0,
             "head_linear_mfma: bad sizes tokens=%d heads=%d k=%d n=%d strides %ld %ld", tokens, heads, K, N, xs_t, xs_h);
  PA_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0, "head_linear_mfma: operands are not 16-byte aligned");
  const int tiles = (N + 15) / 16, steps = (K + 63) / 64;
  const bool whole = whole_stores(y, sizeof(bf16), ys_t, 0) && ys_h % 4 == 0;
  hipStream_t st = (hipStream_t)stream;
#define PA_HL(RM, NT, WAVES)                                                                                               \
  do {                                                                                                                     \
    const long across = (tiles + NT - 1) / NT, down = (tokens + 16 * RM - 1) / (16 * RM);                                  \
    PA_REQUIRE(heads <= 65535 && across * down + turns <= 0x7fffffffL, "head_linear_mfma: %d heads exceed the grid", heads);       \
    hipLaunchKernelGGL((head_linear_mfma_kernel<RM, NT, WAVES>), dim3((unsigned)(across * down + turns), heads),           \
                       dim3(WAVES * kWave), 0, st, (const bf16*)x, (const bf16*)w, (bf16*)y, tokens, K, N, xs_t, xs_h,     \
                       ys_t, ys_h, whole, turn);                                                                                \
  } while (0)
  if (tokens <= 16) {
    if (steps <= 3) PA_HL(1, 1, 2);
    else PA_HL(1, 1, 8);
  } else {
    if (steps <= 3) PA_HL(2, 1, 2);
    else PA_HL(4, 2, 8);
  }
#undef PA_HL
  return check_launch("head_linear_mfma");
}

// y[m, N] (N / 2 for gated pairs) = act(x[m, K] W^T) for up to 16 rows, w in tiles; K a multiple of 8, x and w in 16-byte pieces.
extern "C" int pa_linear_few_act(void* stream, const void* x, const void* w, void* y, int m, int K, int N, int act, float limit, float alpha) {
  if (m == 0) return 0;
  PA_REQUIRE(m > 0 && m <= 16 && K > 0 && N > 0 && K % 8 == 0, "linear_few_act: bad sizes m=%d (up to 16) k=%d n=%d", m, K, N);
  PA_REQUIRE(act >= 0 && act <= 3 && (act < 2 || N % 2 == 0) && (act != 2 || limit > 0.f), "linear_few_act: activation %d over %d outputs, clamp %g",
             act, N, (double)limit);
  PA_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0, "linear_few_act: operands are not 16-byte aligned");
  hipLaunchKernelGGL(linear_few_mfma_kernel, dim3((N + 15) / 16), dim3(512), 0, (hipStream_t)stream, (const bf16*)x, (const bf16*)w, (bf16*)y,
                     m, K, N, whole_stores(y, sizeof(bf16), act >= 2 ? N / 2 : N, act), act, limit, alpha);
  return check_launch("linear_few_act");
}
