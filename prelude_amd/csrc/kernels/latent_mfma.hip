// Attention over a cache of latents on the matrix cores (bfloat16 in, 32-bit scores, softmax and sums).
//
// All heads read the same cached vectors, so the rows of the score matrix are (token, head) pairs: a workgroup
// of four wavefronts owns 64 consecutive rows of one sequence's portion (row = token * heads + head), 16 a
// wavefront, and walks the keys in blocks of 32.  A block is brought into LDS once per workgroup: the vectors as
// they lie in the cache (rows of rank + rot elements, the score's operand), and the first `rank` elements of each
// again transposed ([element][key]: the operand of the weighted sum, whose contraction runs over keys).  The cache
// keeps that transposed copy itself ([pages, rank, page]), written once per token, so both are copied in 16-byte
// pieces, from memory straight into LDS.
//
//   S^T = K Q^T     A = 16 keys x 32 elements from LDS, B = the wavefront's queries, kept in registers
//   O^T = V^T P^T   A = 16 elements x 32 keys from the transposed copy, B = the probabilities just computed
//
// v_mfma_f32_16x16x32_bf16 (lane l, g = l / 16, r = l % 16): A row r, columns 8g..8g+7; B column r, rows 8g..8g+7;
// C column r, rows 4g..4g+3.  A block's 32 keys are two score tiles; row 4a + i of tile t stands for key
// 8a + 4t + i, so lane group g ends up with the scores of keys 8g..8g+7 of its query: packed, they are the B
// operand of the second product as they stand.
//
// Few rows a sequence (single decoded tokens) would leave the chip empty: then the keys are cut into splits of
// `split_keys`, each leaving an unnormalised partial (maximum, sum, weighted sum) that a merge kernel adds up in split
// order; such steps go to latent_attn_decode_kernel below.  (The kernel of portions takes splits too, in grid.z, for a
// caller that asks for it: the two are held against each other that way.)  The sink joins last, as one more term
// exp(sink_h) of the denominator.
#include "common.h"
#include "api.h"

namespace pa {

constexpr float kLog2eL = 1.4426950408889634f;
constexpr int kLmRows = 64;      // query rows a workgroup
constexpr int kLmKeys = 32;      // keys a block
constexpr int kLmPad = 8;        // elements of padding behind an LDS row

// 64 pieces of 16 bytes from memory straight into LDS: lane l's piece lands at `lds_base` + 16 l.  Written as the
// instruction itself: through the compiler's own builtin every later read of LDS first waited for all such loads
// (it cannot tell the two buffers apart), which put the staging in line with the products instead of behind them.
// The kernel waits for them itself (vmcnt 0) before the barrier that publishes a buffer.
__device__ __forceinline__ void load_to_lds_16(const void* src, void* lds_base) {
  const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds_base);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(base), "v"(src) : "memory");
}

// Of a 16-lane group's four rows of sixteen elements, four of one row at each lane's place (lanes 4 i .. 4 i + 3: row i), the lane's column.
__device__ __forceinline__ bf16x4 read_turned(const bf16* at) {
  typedef short short4v __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v*)at));
}

__device__ __forceinline__ f32x4 mfma16l(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Which of eight keys from key0 on lie in [lo, end), as a mask over their bfloat16 values.  A key that is not seen has the
// probability 0, but its place may hold anything (what a page's earlier owner left, a page that now is another request's),
// and 0 times NaN is NaN: blocks at an end of a range take such values out before the product.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 keys_seen(int key0, int lo, int end) {
  u32x4 m;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int a = key0 + 2 * i, b = a + 1;
    m[i] = (a >= lo && a < end ? 0xffffu : 0u) | (b >= lo && b < end ? 0xffff0000u : 0u);
  }
  return m;
}

__device__ __forceinline__ bf16x8 only(bf16x8 v, u32x4 m) { return __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, v) & m); }

// RT: value tiles of 16 elements held in registers (rank <= 16 RT); QS: steps of 32 elements of a query held in
// registers (rank + rot <= 32 QS).
template <int RT, int QS>
__global__ __launch_bounds__(256) void latent_attn_mfma_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ cache, const bf16* __restrict__ cache_t,
    const float* __restrict__ sink, const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out,
    float* __restrict__ ws, int nh, int rank, int rot, int page_size, int window, float scale, int split_keys,
    int n_splits) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int dk = rank + rot;
  const int dk_steps = (dk + 31) / 32;
  const int k_stride = dk_steps * 32 + kLmPad;                 // elements
  const int v_tiles = (rank + 15) / 16;
  constexpr int v_stride = kLmKeys + kLmPad;

  const int seq = seq_ids ? seq_ids[blockIdx.y] : blockIdx.y;
  const int q0 = cu_q[seq], qn = cu_q[seq + 1] - q0;
  const int rows = qn * nh;
  const int rb = blockIdx.x * kLmRows;
  if (rb >= rows) return;
  const int ctx = context_lens[seq];
  const int p0 = ctx - qn;                                     // position of the portion's first token
  const int* table = block_table + (size_t)seq * table_stride;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;

  // this lane's query row (clamped: rows past the end repeat the last one and are not stored)
  const int row = rb + wave * 16 + r;
  const bool row_ok = row < rows;
  const int rowc = row_ok ? row : rows - 1;
  const int tq = rowc / nh, head = rowc % nh;
  const int pos = p0 + tq;
  const int lo_row = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;

  // keys the workgroup walks: up to its last row's position, from its first row's window edge, inside its split
  const int last_row = (rb + kLmRows - 1 < rows ? rb + kLmRows - 1 : rows - 1);
  const int hi_wg = p0 + last_row / nh;
  const int first_pos = p0 + rb / nh;
  int lo_wg = (window > 0 && first_pos - window + 1 > 0) ? first_pos - window + 1 : 0;
  int end_wg = hi_wg + 1;
  if (n_splits > 1) {
    const int s0 = blockIdx.z * split_keys;
    lo_wg = lo_wg > s0 ? lo_wg : s0;
    end_wg = end_wg < s0 + split_keys ? end_wg : s0 + split_keys;
  }
  const int lo_seen = lo_wg;
  lo_wg = (lo_wg / kLmKeys) * kLmKeys;                         // blocks stand at multiples of 32 keys

  // queries: B operand, column r = this lane's row, rows 8g..8g+7 of every step of 32 elements
  bf16x8 qf[QS];
  {
    const bf16* qr = q + ((size_t)(q0 + tq) * nh + head) * dk;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      const int d = 32 * s + 8 * g;
      bf16x8 v = {};
      if (d + 8 <= dk) v = *reinterpret_cast<const bf16x8*>(qr + d);
      qf[s] = v;
    }
  }
  f32x4 o[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float c = scale * kLog2eL;
  const bool wave_active = rb + wave * 16 < rows;              // a wavefront without rows of its own only helps staging

  // Staging goes from memory straight into LDS (no registers in between: with the queries and the output tiles a
  // wavefront holds, staged pieces parked in registers were waited for one by one).  One such load fills 64
  // consecutive 16-byte pieces of LDS, a piece a lane, from 64 addresses of the lanes' own; the two regions are
  // laid out piece by piece: rows of k_pieces (a row's pieces and one of padding), then the transposed copy's rows
  // of five (four runs of 8 keys and one of padding).  Pieces of padding, keys past the range and pages given back
  // are loaded from clamped addresses: what they bring is masked, or taken out before the product.  Two buffers:
  // the next block's loads are in flight while this block is worked on.
  const int k_pieces = dk_steps * 4 + 1;
  const int k_loads = (kLmKeys * k_pieces + 63) / 64, v_loads = (v_tiles * 16 * 5 + 63) / 64;
  const int buf_elems = (k_loads + v_loads) * 512;             // 64 pieces of 8 elements a load
  const int ch_last = dk / 8 - 1;
  // Where this lane's piece of each load lies does not change from block to block: piece i = 64 * load + lane of
  // the rows is key i / k_pieces, piece i % k_pieces; of the transposed copy element i / 5, run i % 5 of 8 keys (the
  // fifth is padding).  So each load's share of the address is worked out once, before the first block: the offset
  // inside the block's run of 8 keys (24 bits) and which of the block's four runs it is (the bits above).  A block
  // then costs a load a choice among four bases and an addition.  (Pages hold multiples of 8 keys, so a run lies in
  // one page.  Pieces of padding, elements and keys that do not exist take the place of ones that do.)
  constexpr int KS = ((kLmKeys * (QS * 4 + 1) + 63) / 64 + 3) / 4;      // loads of rows a wavefront, at most
  constexpr int VS = ((RT * 16 * 5 + 63) / 64 + 3) / 4;                 // loads of the copy a wavefront, at most
  unsigned kinfo[KS], vinfo[VS];
#pragma unroll
  for (int sl = 0; sl < KS; ++sl) {
    const int i = (wave + 4 * sl) * 64 + lane;
    int key = i / k_pieces, ch = i % k_pieces;
    key = key < kLmKeys ? key : kLmKeys - 1;
    ch = ch < ch_last ? ch : ch_last;
    kinfo[sl] = (unsigned)((key & 7) * dk + 8 * ch) | ((unsigned)(key >> 3) << 24);
  }
#pragma unroll
  for (int sl = 0; sl < VS; ++sl) {
    const int i = (wave + 4 * sl) * 64 + lane;
    int vrow = i / 5, j = i % 5;
    vrow = vrow < rank ? vrow : rank - 1;
    j = j < 4 ? j : 0;
    vinfo[sl] = (unsigned)(vrow * page_size) | ((unsigned)j << 24);
  }
  const int last = ctx - 1;                                      // the sequence's last key
  auto issue_block = [&](int b0, bf16* buf) {
    const int rel_last = last - b0;                              // >= 0: the block holds a key of the range
    // where the block's four runs of 8 keys start, in the cache and in the copy (the same for every lane); a run past
    // the sequence takes the place of its last one
    const bf16* krun[4];
    const bf16* vrun[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int kc = 8 * j <= rel_last ? b0 + 8 * j : (last & ~7);
      const int at = kc / page_size;
      const int page = table[at];
      const size_t pg = page >= 0 ? page : 0, place = kc - at * page_size;
      krun[j] = cache + (pg * page_size + place) * dk;
      vrun[j] = cache_t + pg * rank * page_size + place;
    }
#pragma unroll
    for (int sl = 0; sl < KS; ++sl) {
      const int sI = wave + 4 * sl;
      if (sI < k_loads) {
        const unsigned j = kinfo[sl] >> 24;
        const bf16* base = j == 0 ? krun[0] : (j == 1 ? krun[1] : (j == 2 ? krun[2] : krun[3]));
        load_to_lds_16(base + (kinfo[sl] & 0xffffffu), buf + (size_t)sI * 512);
      }
    }
#pragma unroll
    for (int sl = 0; sl < VS; ++sl) {
      const int sI = wave + 4 * sl;
      if (sI < v_loads) {
        const unsigned j = vinfo[sl] >> 24;
        const bf16* base = j == 0 ? vrun[0] : (j == 1 ? vrun[1] : (j == 2 ? vrun[2] : vrun[3]));
        load_to_lds_16(base + (vinfo[sl] & 0xffffffu), buf + (size_t)(k_loads + sI) * 512);
      }
    }
  };

  const int wave_pos_min = __shfl(pos, 0, kWave);              // the wavefront's rows ascend: its first row sees least,
  const int wave_lo_max = __shfl(lo_row, 15, kWave);           // its last row's window starts last
  bf16* const buf0 = reinterpret_cast<bf16*>(lds_raw);
  if (lo_wg < end_wg) issue_block(lo_wg, buf0);
  int it = 0;
  for (int b0 = lo_wg; b0 < end_wg; b0 += kLmKeys, ++it) {
    bf16* const cur = buf0 + (it & 1) * buf_elems;
    __builtin_amdgcn_s_waitcnt(0);                             // this wavefront's share of the block has landed
    __syncthreads();                                           // ... and everyone's; all are done with the other buffer
    if (b0 + kLmKeys < end_wg) issue_block(b0 + kLmKeys, buf0 + ((it + 1) & 1) * buf_elems);
    // values in front of the window and behind the sequence, which may be anything (the same for the whole workgroup; in LDS, where
    // it costs no registers; keys of the sequence behind this workgroup's are its own and meet zeros)
    if (b0 < lo_seen || b0 + kLmKeys > ctx) {
      for (int i = threadIdx.x; i < v_tiles * 16 * 4; i += 256) {
        bf16x8* v = reinterpret_cast<bf16x8*>(cur + k_loads * 512 + (i / 4) * v_stride + 8 * (i % 4));
        *v = only(*v, keys_seen(b0 + 8 * (i % 4), lo_seen, ctx));
      }
      __syncthreads();
    }
    if (!wave_active) continue;
    const bf16* k_lds = cur;
    const bf16* v_lds = cur + k_loads * 512;
    // ---- scores of 32 keys for this wavefront's 16 rows ----
    // Operands are read from LDS in batches ahead of the products that use them (a wavefront is alone on its SIMD:
    // a read waited for right before its product costs the LDS's latency every time), and the two tiles' chains of
    // dependent products run interleaved.
    f32x4 s[2];
    s[0] = f32x4{0.f, 0.f, 0.f, 0.f};
    s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    {
      const bf16* kr0 = k_lds + (8 * (r / 4) + (r % 4)) * k_stride + 8 * g;
      const bf16* kr1 = kr0 + 4 * k_stride;
      constexpr int kBatch = 6;
#pragma unroll
      for (int k0 = 0; k0 < QS; k0 += kBatch) {
        bf16x8 ka[kBatch], kb[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          // (offsets known when compiled: a step past the latent's own width reads on into the buffer -- the rows
          // are followed by the transposed copy, so it stays inside -- and is not multiplied)
          const int ks = k0 + j < QS ? k0 + j : QS - 1;
          ka[j] = *reinterpret_cast<const bf16x8*>(kr0 + 32 * ks);
          kb[j] = *reinterpret_cast<const bf16x8*>(kr1 + 32 * ks);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
          if (k0 + j < QS && k0 + j < dk_steps) {
            s[0] = mfma16l(ka[j], qf[k0 + j], s[0]);
            s[1] = mfma16l(kb[j], qf[k0 + j], s[1]);
          }
        }
      }
    }
    // ---- mask, running maximum, probabilities ----
    // (a block that every row of the wavefront sees whole, which is most of them, skips the mask)
    float bm = -INFINITY;
    if (b0 + kLmKeys - 1 <= wave_pos_min && b0 >= wave_lo_max && b0 + kLmKeys <= end_wg) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) bm = fmaxf(bm, s[t][i]);
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kidx = b0 + 8 * g + 4 * t + i;
          const bool ok = kidx <= pos && kidx >= lo_row && kidx < end_wg;
          s[t][i] = ok ? s[t][i] : -INFINITY;
          bm = fmaxf(bm, s[t][i]);
        }
    }
    bm = fmaxf(bm, __shfl_xor(bm, 16, kWave));
    bm = fmaxf(bm, __shfl_xor(bm, 32, kWave));
    // The exponentials are taken against a reference that follows the running maximum lazily: it moves, and the
    // sums are rescaled, only when a score exceeds it by 2^8 (then probabilities stay below 256, which 32-bit sums
    // and bfloat16 operands hold as well as values below 1); after the first blocks that is rare.
    const bool move = m == -INFINITY || (bm - m) * c > 8.f;
    const float m_new = move ? bm : m;
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float shift = -m_use * c;
    const float alpha = move ? __builtin_amdgcn_exp2f(fmaf(m, c, shift)) : 1.0f;
    float psum = 0.f;
    bf16x8 pf;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][i], c, shift));       // 2^-inf = 0 for masked keys
        psum += p;
        pf[4 * t + i] = (bf16)p;
      }
    l = l * alpha + psum;
    m = m_new;
    // ---- weighted sum: O^T += V^T P^T ----
    // (the sums are rescaled only in blocks where some row's maximum moved: early ones, and rarely later)
    const bool rescale = __any(alpha != 1.0f);
    {
      const bf16* vr = v_lds + r * v_stride + 8 * g;
      constexpr int vBatch = 8;
#pragma unroll
      for (int t0 = 0; t0 < RT; t0 += vBatch) {
        if (t0 < v_tiles) {
          bf16x8 vf[vBatch];
#pragma unroll
          for (int j = 0; j < vBatch; ++j) {
            const int t = t0 + j < RT ? t0 + j : RT - 1;
            vf[j] = *reinterpret_cast<const bf16x8*>(vr + 16 * (t < v_tiles ? t : 0) * v_stride);
          }
#pragma unroll
          for (int j = 0; j < vBatch; ++j) {
            if (t0 + j < RT && t0 + j < v_tiles) {
              if (rescale) o[t0 + j] *= alpha;
              o[t0 + j] = mfma16l(vf[j], pf, o[t0 + j]);
            }
          }
        }
      }
    }
  }

  // ---- the row's sum over its four lanes; then the sink and the division, or the partial for the merge ----
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  if (!row_ok) return;
  const float mn = m * scale;                                  // the maximum in the exponent's own unit
  if (n_splits > 1) {
    // (splits are for sequences of one token: the partial's row is the sequence's place in the launch and the head)
    const size_t part = ((size_t)blockIdx.y * nh + head) * n_splits + blockIdx.z;
    if (g == 0) *reinterpret_cast<f32x2*>(ws + (size_t)gridDim.y * nh * n_splits * rank + 2 * part) = f32x2{mn, l};
    float* w = ws + part * rank;
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (16 * t + 4 * g < rank) *reinterpret_cast<f32x4*>(w + 16 * t + 4 * g) = o[t];
    return;
  }
  float a = 1.f;
  if (sink) {
    const float sk = sink[head];
    const float top = fmaxf(mn, sk);
    a = expf(mn - top);
    l = l * a + expf(sk - top);
  }
  const float inv = a / l;
  bf16* orow = out + ((size_t)(q0 + tq) * nh + head) * rank;
#pragma unroll
  for (int t = 0; t < RT; ++t)
    if (t < v_tiles) {
      const int d = 16 * t + 4 * g;
      if (d + 4 <= rank) {
        bf16x4 v = {(bf16)(o[t][0] * inv), (bf16)(o[t][1] * inv), (bf16)(o[t][2] * inv), (bf16)(o[t][3] * inv)};
        *reinterpret_cast<bf16x4*>(orow + d) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (d + i < rank) orow[d + i] = (bf16)(o[t][i] * inv);
      }
    }
}

// Steps of single tokens: a sequence brings only `heads` rows, one tile of 16 for 16 heads.  A workgroup is a split of the keys of one
// sequence and 16 heads, and its four wavefronts share the work both ways: of a block of 64 keys each takes the scores of 16
// keys, and, the probabilities exchanged through LDS, the weighted sum of a quarter of the latent's elements over all 64.
// What bounds it is memory, so the latents come once: a block's rows, from memory straight into LDS, 16 keys a wavefront, are the score's
// operand as they lie, and the sum's, whose contraction runs over keys, by LDS reads that hand four keys' elements to
// sixteen lanes turned (ds_read_b64_tr_b16).  A block is 72 KB, two workgroups a compute unit, one of which asks while the other
// multiplies.  With the merge, us, both copies of the cache read into registers / like this: 8 sequences of 4,097 keys 26.5 / 20.0, 32 and
// 64 of 4,096 65 / 37.5 and 125 / 70 (302 MB: 4.9 TB/s), one of 32,768 36.3 / 20.5, of 4,097 15.0 / 13.1, four of 150 12.6 / 11.5.  Two
// blocks on their way in one workgroup a compute unit are no faster: 20.2 at best, and 39 and 76.
// In LDS the rows lie one behind the other (brought by kilobytes of one row and the next: eight keys by whole lines each took 41 us
// for 32 sequences of 4,096 keys, 39 like this), the 16-byte pieces of each exchanged by the key's number (latent_turn), so that
// sixteen keys' pieces of one place, and eight keys' pairs of neighbouring ones, lie in different banks.
// Lane (g, r) of a step of 64 elements holds elements 16 g .. 16 g + 15 of key r, the first eight for one product and the
// others for the next, and the queries lie in the same order.
// Grid (sequences, splits, tiles of 16 heads).
constexpr int kLdKeys = 64;      // keys a block
__device__ __forceinline__ int latent_turn(int key) { return (key >> 2 & 1) | (key >> 1 & 1) << 1 | (key >> 3 & 1) << 2; }

template <int QS>
struct LatentLds {
  static constexpr int kPieces = QS * 4;                         // 16-byte pieces a key
  static constexpr int kPRow = kLdKeys + 8;                      // a row of probabilities: 16 bytes of padding
  __align__(16) bf16 keys[kLdKeys][kPieces][8];
  __align__(16) bf16 ps[2][16][kPRow];
  float tops[4][16];
};

template <int RT, int QS>
__global__ __launch_bounds__(256, 2) void latent_attn_decode_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ cache, const int* __restrict__ block_table, int table_stride,
    const int* __restrict__ seq_ids, const int* __restrict__ cu_q, const int* __restrict__ context_lens, float* __restrict__ ws, int nh,
    int rank, int rot, int page_size, int window, float scale, int split_keys, int n_splits) {
  typedef LatentLds<QS> Lds;
  constexpr int kPieces = Lds::kPieces, kPairs = QS / 2;         // steps of 64 elements
  constexpr int kTiles = RT / 4;                                 // tiles of 16 elements a wavefront
  constexpr int kBases = kTiles < 4 ? kTiles : 4;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  Lds& lds = *reinterpret_cast<Lds*>(lds_raw);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int z = blockIdx.y;
  const int seq = seq_ids ? seq_ids[blockIdx.x] : blockIdx.x;
  const int tok = cu_q[seq];
  const int pos = context_lens[seq] - 1;
  const int dk = rank + rot;
  const int* table = block_table + (size_t)seq * table_stride;
  const int head0 = blockIdx.z * 16;
  const int head = head0 + r < nh ? head0 + r : nh - 1;
  const int lo_row = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  int lo = z * split_keys, end = lo + split_keys;
  lo = lo > lo_row ? lo : lo_row;
  end = end < pos + 1 ? end : pos + 1;
  const int b_first = (lo / kLdKeys) * kLdKeys, last = end - 1;

  f32x4 o[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float c = scale * kLog2eL;

  if (lo < end) {                                                // (the same for the whole workgroup)
    // Where lane r's key of this wavefront's sixteen lies, in rows of the cache; a key past the range takes the place of the last
    // one inside it (masked).
    auto row_of = [&](int b0) {
      int kidx = b0 + 16 * wave + r;
      kidx = kidx < last ? kidx : last;
      const int at = kidx / page_size, page = table[at];
      return (page >= 0 ? page : 0) * page_size + (kidx - at * page_size);
    };
    const bool whole = dk == 64 * kPairs;
    auto ask = [&](int row) {
#pragma unroll
      for (int i = 0; i < kPieces / 4; ++i) {                    // the wavefront's rows in turn, 64 pieces a load
        const int begin = i * kWave / kPieces;                   // a row of 72 pieces or the next one, else whichever it is
        const int key = kPieces > kWave ? begin + (i * kWave + lane >= (begin + 1) * kPieces) : (i * kWave + lane) / kPieces;
        int at;
        if constexpr (kPieces > kWave) {
          const int one = __builtin_amdgcn_readlane(row, begin), two = __builtin_amdgcn_readlane(row, begin < 15 ? begin + 1 : 15);
          at = key == begin ? one : two;
        } else {
          at = __shfl(row, key, kWave);
        }
        const int piece = (i * kWave + lane - key * kPieces) ^ latent_turn(key);
        const int d = whole || 8 * piece < dk ? 8 * piece : 0;   // elements that do not exist: others, not counted
        load_to_lds_16(cache + ((size_t)(unsigned)at * dk + d), &lds.keys[16 * wave][0][0] + i * kWave * 8);
      }
    };
    const int first = row_of(b_first);
    bf16x8 qf[kPairs][2];
    {
      const bf16* qr = q + ((size_t)tok * nh + head) * dk;
#pragma unroll
      for (int s = 0; s < kPairs; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int d = 64 * s + 16 * g + 8 * h;
          qf[s][h] = *reinterpret_cast<const bf16x8*>(qr + (d < dk ? d : 0));
        }
    }
    __builtin_amdgcn_sched_barrier(0);                           // the queries are on their way while the page number comes
    ask(first);
    if (!whole) {                                                // elements that do not exist are zeros: what a key brings there does not count
#pragma unroll
      for (int s = 0; s < kPairs; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (64 * s + 16 * g + 8 * h >= dk) qf[s][h] = bf16x8{};
    }
    // the keys of the scores: a base for either half of a step; of the sums: one for every tile of four, and every half of a lane's eight keys
    const bf16* kb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) kb[h] = lds.keys[16 * wave + r][(2 * g + h) ^ latent_turn(r)];
    const bf16* vb[2][kBases];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int key = 8 * g + 4 * h + r / 4;
#pragma unroll
      for (int t = 0; t < kBases; ++t) vb[h][t] = lds.keys[key][(2 * (wave * kTiles + t) + r % 4 / 2) ^ latent_turn(key)] + r % 2 * 4;
    }
    for (int b0 = b_first; b0 < end; b0 += kLdKeys) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const bool more = b0 + kLdKeys < end;
      const int next = more ? row_of(b0 + kLdKeys) : 0;
      // ---- scores of 16 keys: two chains of dependent products ----
      f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < kPairs; ++s) {
        sa = mfma16l(*reinterpret_cast<const bf16x8*>(kb[0] + 64 * s), qf[s][0], sa);
        sb = mfma16l(*reinterpret_cast<const bf16x8*>(kb[1] + 64 * s), qf[s][1], sb);
      }
      // ---- the block's maximum over all four wavefronts, probabilities ----
      float sc[4], bm = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kidx = b0 + 16 * wave + 4 * g + i;
        sc[i] = kidx >= lo && kidx < end ? sa[i] + sb[i] : -INFINITY;
        bm = fmaxf(bm, sc[i]);
      }
      bm = fmaxf(bm, __shfl_xor(bm, 16, kWave));
      bm = fmaxf(bm, __shfl_xor(bm, 32, kWave));
      if (g == 0) lds.tops[wave][r] = bm;
      __syncthreads();
      bm = fmaxf(fmaxf(lds.tops[0][r], lds.tops[1][r]), fmaxf(lds.tops[2][r], lds.tops[3][r]));
      // (against a reference that follows the maximum lazily, as above; the same in every wavefront)
      const bool move = m == -INFINITY || (bm - m) * c > 8.f;
      const float m_new = move ? bm : m;
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float shift = -m_use * c;
      const float alpha = move ? __builtin_amdgcn_exp2f(fmaf(m, c, shift)) : 1.0f;
      float psum = 0.f;
      // a probability as two bfloat16 numbers, the second what the first leaves: the products wait for memory either way (a
      // microsecond of 28), and the result is off by 1.65e-3 of its norm, what its own rounding to bfloat16 costs, instead of
      // the 1.8e-3 to 2.1e-3 of probabilities rounded once
      bf16x4 pv, pl;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[i], c, shift));   // 2^-inf = 0 for masked keys
        psum += p;
        pv[i] = (bf16)p;
        pl[i] = (bf16)(p - (float)pv[i]);
      }
      l = l * alpha + psum;
      m = m_new;
      *reinterpret_cast<bf16x4*>(&lds.ps[0][r][16 * wave + 4 * g]) = pv;
      *reinterpret_cast<bf16x4*>(&lds.ps[1][r][16 * wave + 4 * g]) = pl;
      __syncthreads();
      // ---- weighted sum of this wavefront's elements over the block ----
      bf16x8 p[2][2];
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int step = 0; step < 2; ++step) p[part][step] = *reinterpret_cast<const bf16x8*>(&lds.ps[part][r][32 * step + 8 * g]);
      const bool edge = b0 < lo || b0 + kLdKeys > end;           // (the same for the whole workgroup)
      const bool rescale = __any(alpha != 1.0f);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        if (rescale) o[t] *= alpha;
        bf16x8 vf[2];
#pragma unroll
        for (int step = 0; step < 2; ++step) {
          bf16x4 half[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) half[h] = read_turned(vb[h][t % kBases] + 32 * step * kPieces * 8 + t / kBases * 64);
          vf[step] = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
          if (edge) {
            const int k0 = b0 + 32 * step + 8 * g;
#pragma unroll
            for (int i = 0; i < 8; ++i) vf[step][i] = k0 + i >= lo && k0 + i < end ? vf[step][i] : (bf16)0.f;
          }
        }
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int step = 0; step < 2; ++step) o[t] = mfma16l(vf[step], p[part][step], o[t]);
      }
      // (the next block's probabilities are written behind everyone's reads of these: the barriers of its rows and of its maxima do)
      if (more) {
        __syncthreads();                                         // everyone has read this block
        ask(next);
      }
    }
    // the head's sum over its lanes and wavefronts, in their order
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    __syncthreads();
    if (g == 0) lds.tops[wave][r] = l;
    __syncthreads();
    l = (lds.tops[0][r] + lds.tops[1][r]) + (lds.tops[2][r] + lds.tops[3][r]);
  }
  if (head0 + r >= nh) return;
  const size_t part = ((size_t)blockIdx.x * nh + head) * n_splits + z;
  if (wave == 0 && g == 0) *reinterpret_cast<f32x2*>(ws + (size_t)gridDim.x * nh * n_splits * rank + 2 * part) = f32x2{m * scale, l};
  float* w = ws + part * rank;
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const int d = 16 * (wave * kTiles + t) + 4 * g;
    if (d < rank) *reinterpret_cast<f32x4*>(w + d) = o[t];
  }
}

// out[row] = sum over the splits' partials, each scaled by exp(its maximum - the largest), then the sink.  ws holds every
// row's weighted sums [rows][splits][rank] (rank is a multiple of 8: whole fours stay aligned) and behind them the
// (maximum, sum) pairs [rows][splits][2].  A workgroup takes
// 64 elements of a row: the splits' factors are worked out once (in LDS), its four wavefronts take the splits in turn,
// eight loads in flight, and are added in their order.  (With a workgroup a whole row, the rows of few sequences left most
// of the chip idle while each walked all splits: 5.5 us instead of 7.9 for 8 sequences in 20 splits then and 40 now; with one of
// 32,768 keys in 512 splits attention and merge together went from 84 to 36.)
constexpr int kMergeMaxSplits = 4096;
__global__ __launch_bounds__(256) void latent_attn_merge_kernel(const float* __restrict__ ws, const float* __restrict__ sink,
                                                               const int* __restrict__ seq_ids, const int* __restrict__ cu_q,
                                                               bf16* __restrict__ out, int nh, int rank, int n_splits) {
  __shared__ float factor[kMergeMaxSplits];
  __shared__ float scratch[16];
  __shared__ float sums[4][kWave];
  const int row = blockIdx.x;                                  // (place in the launch) * heads + head
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const f32x2* ml = reinterpret_cast<const f32x2*>(ws + (size_t)gridDim.x * n_splits * rank) + (size_t)row * n_splits;
  float top = -INFINITY;
  for (int z = threadIdx.x; z < n_splits; z += 256) top = fmaxf(top, ml[z][0]);
  top = wave_max(top);
  if (lane == 0) scratch[wave] = top;
  __syncthreads();
  top = fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3]));
  const float sk = sink ? sink[row % nh] : -INFINITY;
  top = fmaxf(top, sk);
  float lpart = 0.f;
  for (int z = threadIdx.x; z < n_splits; z += 256) {
    const f32x2 v = ml[z];
    const float f = v[0] == -INFINITY ? 0.f : expf(v[0] - top);
    factor[z] = f;
    lpart += f * v[1];
  }
  float l = block_sum(lpart, scratch);                         // (its barriers also publish the factors)
  if (sink) l += expf(sk - top);
  const int d = blockIdx.y * kWave + lane, dc = d < rank ? d : rank - 1;
  const float* w = ws + (size_t)row * n_splits * rank + dc;
  float acc = 0.f;
  int z = wave;
  for (; z + 28 < n_splits; z += 32) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = w[(size_t)(z + 4 * j) * rank];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += v[j] * factor[z + 4 * j];
  }
  for (; z < n_splits; z += 4) acc += w[(size_t)z * rank] * factor[z];
  sums[wave][lane] = acc;
  __syncthreads();
  if (wave || d >= rank) return;
  const int seq = seq_ids ? seq_ids[row / nh] : row / nh;
  out[((size_t)cu_q[seq] * nh + row % nh) * rank + d] = (bf16)(((sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane])) / l);
}

template <int RT, int QS>
static int launch_latent_mfma(hipStream_t st, dim3 grid, size_t lds, const bf16* q, const bf16* cache, const bf16* cache_t, const float* sink,
                              const int* block_table, int table_stride, const int* seq_ids, const int* cu_q,
                              const int* context_lens, bf16* out, float* ws, int nh, int rank, int rot, int page_size,
                              int window, float scale, int split_keys, int n_splits) {
  static bool raised = false;
  if (!raised) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attn_mfma_kernel<RT, QS>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return pa::fail("latent_attn_mfma: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = true;
  }
  hipLaunchKernelGGL((latent_attn_mfma_kernel<RT, QS>), grid, dim3(256), lds, st, q, cache, cache_t, sink, block_table, table_stride,
                     seq_ids, cu_q, context_lens, out, ws, nh, rank, rot, page_size, window, scale, split_keys, n_splits);
  return 0;
}

template <int RT, int QS>
static int launch_latent_decode(hipStream_t st, dim3 grid, const bf16* q, const bf16* cache, const int* block_table, int table_stride,
                                const int* seq_ids, const int* cu_q, const int* context_lens, float* ws, int nh, int rank, int rot,
                                int page_size, int window, float scale, int split_keys, int n_splits) {
  static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attn_decode_kernel<RT, QS>),
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(LatentLds<QS>));
  if (allowed != hipSuccess) return pa::fail("latent_attn_decode: %zu bytes of LDS refused: %s", sizeof(LatentLds<QS>), hipGetErrorString(allowed));
  hipLaunchKernelGGL((latent_attn_decode_kernel<RT, QS>), grid, dim3(256), sizeof(LatentLds<QS>), st, q, cache, block_table, table_stride,
                     seq_ids, cu_q, context_lens, ws, nh, rank, rot, page_size, window, scale, split_keys, n_splits);
  return check_launch("latent_attn_decode");
}

static size_t latent_mfma_lds(int rank, int rot) {
  const int dk_steps = (rank + rot + 31) / 32, v_tiles = (rank + 15) / 16;
  const int k_loads = (kLmKeys * (dk_steps * 4 + 1) + 63) / 64, v_loads = (v_tiles * 16 * 5 + 63) / 64;
  return (size_t)2 * (k_loads + v_loads) * 1024;               // two buffers of whole 64-piece loads
}

}  // namespace pa

using namespace pa;

// Sizes the matrix-core kernel takes: 16-byte rows, at most 512 + 64 elements, pages of a multiple of 8 keys.
extern "C" int pa_latent_attn_mfma_supports(int rank, int rot, int page_size) {
  return rank > 0 && rot >= 0 && rank % 8 == 0 && rot % 8 == 0 && rank <= 512 && rot <= 64 && page_size > 0 && page_size % 8 == 0 &&
         page_size <= 16384 &&   // (an element's offset in the transposed copy, rank * page_size, is kept in 24 bits)
         latent_mfma_lds(rank, rot) <= 160 * 1024;
}

// 32-bit words of workspace for `n_seqs` sequences of one token in `n_splits` splits
extern "C" long pa_latent_attn_mfma_workspace(int n_seqs, int nh, int rank, int n_splits) {
  return n_splits > 1 ? (long)n_seqs * nh * n_splits * (rank + 2) : 0;
}

// q [tokens, heads, rank + rot], cache [pages, page, rank + rot] and its latents transposed, cache_t [pages, rank, page]
// -> out [tokens, heads, rank] for the sequences seq_ids[0..n_seqs) (null: sequences
// 0..n_seqs), each with cu_q[s+1] - cu_q[s] tokens ending at context_lens[s]; max_q_len bounds their tokens.
// n_splits > 1 (sequences of one token only): the keys in splits of split_keys, partials in ws, merged here; a split is
// a workgroup of the staged kernel, or with `wave_splits` of the kernel that reads the cache directly.
extern "C" int pa_latent_attn_mfma(void* stream, const void* q, const void* cache, const void* cache_t, const float* sink, const int* block_table,
                                   int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens, void* out,
                                   void* ws, int n_seqs, int max_q_len, int nh, int rank, int rot, int page_size,
                                   int window, float scale, int split_keys, int n_splits, int wave_splits) {
  if (n_seqs == 0) return 0;
  PA_REQUIRE(pa_latent_attn_mfma_supports(rank, rot, page_size), "latent_attn_mfma: a latent of %d + %d is not a size it takes", rank, rot);
  PA_REQUIRE(n_seqs > 0 && max_q_len > 0 && nh > 0 && table_stride > 0 && window >= 0,
             "latent_attn_mfma: bad sizes seqs=%d q=%d heads=%d stride=%d window=%d", n_seqs, max_q_len, nh, table_stride, window);
  PA_REQUIRE(cache && cache_t, "latent_attn_mfma: needs the cache and its transposed copy");
  PA_REQUIRE((uintptr_t)ws % 16 == 0, "latent_attn_mfma: the workspace is not 16-byte aligned");
  PA_REQUIRE(scale > 0.f, "latent_attn_mfma: a scale of %g is not positive", (double)scale);
  PA_REQUIRE(n_splits <= kMergeMaxSplits, "latent_attn_mfma: %d splits are more than the %d the merge takes", n_splits, kMergeMaxSplits);
  PA_REQUIRE(n_splits >= 1 && (n_splits == 1 || (split_keys > 0 && split_keys % kLmKeys == 0 && ws && max_q_len == 1)),
             "latent_attn_mfma: %d splits of %d keys need a workspace, whole blocks and sequences of one token", n_splits, split_keys);
  hipStream_t st = (hipStream_t)stream;
  if (n_splits > 1 && wave_splits) {
    // sequences of one token: operands straight from the cache, then the merge
    const int head_tiles = (nh + 15) / 16;
    PA_REQUIRE(n_seqs <= 0x7fffffff && head_tiles <= 65535, "latent_attn_mfma: %d sequences or %d heads exceed the grid", n_seqs, nh);
    PA_REQUIRE(n_splits <= 65535 && split_keys % kLdKeys == 0, "latent_attn_mfma: splits of %d keys are no whole blocks of %d", split_keys, kLdKeys);
    dim3 grid(n_seqs, n_splits, head_tiles);
    int e;
#define PA_LD(RT, QS)                                                                                                                  \
  e = launch_latent_decode<RT, QS>(st, grid, (const bf16*)q, (const bf16*)cache, block_table, table_stride, seq_ids, cu_q, context_lens, \
                                   (float*)ws, nh, rank, rot, page_size, window, scale, split_keys, n_splits)
    if (rank <= 64) PA_LD(4, 4);
    else if (rank <= 128) PA_LD(8, 6);
    else if (rank <= 256) PA_LD(16, 10);
    else PA_LD(32, 18);
#undef PA_LD
    if (e) return e;
    hipLaunchKernelGGL(latent_attn_merge_kernel, dim3(n_seqs * nh, (rank + kWave - 1) / kWave), dim3(256), 0, st, (const float*)ws, sink,
                       seq_ids, cu_q, (bf16*)out, nh, rank, n_splits);
    return check_launch("latent_attn_merge");
  }
  const long tiles = ((long)max_q_len * nh + kLmRows - 1) / kLmRows;
  PA_REQUIRE(tiles <= 0x7fffffffL && n_seqs <= 65535 && n_splits <= 65535, "latent_attn_mfma: the grid %ld x %d x %d is too large", tiles,
             n_seqs, n_splits);
  dim3 grid((unsigned)tiles, n_seqs, n_splits);
  const size_t lds = latent_mfma_lds(rank, rot);
  int rc;
#define PA_LM(RT, QS)                                                                                                  \
  rc = launch_latent_mfma<RT, QS>(st, grid, lds, (const bf16*)q, (const bf16*)cache, (const bf16*)cache_t, sink, block_table, table_stride,  \
                                  seq_ids, cu_q, context_lens, (bf16*)out, (float*)ws, nh, rank, rot, page_size, window, \
                                  scale, split_keys, n_splits)
  if (rank <= 64) PA_LM(4, 4);
  else if (rank <= 128) PA_LM(8, 6);
  else if (rank <= 256) PA_LM(16, 10);
  else PA_LM(32, 18);
#undef PA_LM
  if (rc) return rc;
  if (int e = check_launch("latent_attn_mfma")) return e;
  if (n_splits > 1) {
    hipLaunchKernelGGL(latent_attn_merge_kernel, dim3(n_seqs * nh, (rank + kWave - 1) / kWave), dim3(256), 0, st, (const float*)ws, sink,
                       seq_ids, cu_q, (bf16*)out, nh, rank, n_splits);
    return check_launch("latent_attn_merge");
  }
  return 0;
}
