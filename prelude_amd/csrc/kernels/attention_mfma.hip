// Paged causal attention on the matrix cores (bfloat16 in, 32-bit softmax and
// accumulation), in two kernels that share their inner step:
//
//   attn_decode  -- one query token per sequence; the keys of a sequence are
//                   cut into splits of a fixed number of keys, each workgroup
//                   reduces one split, a second kernel merges the splits.
//   attn_prefill -- portions of several tokens; a wavefront owns 16 tokens of
//                   up to four query heads that share a KV head and walks the
//                   keys they may see.
//
// Both compute S^T = K Q^T and O^T = V^T P^T with v_mfma_f32_16x16x32_bf16, so
// that a query is a column (lane % 16) in the scores and in the output alike:
// the running maximum, the sum and the rescaling stay in the lane, and the
// probabilities leave the first product in exactly the register layout the
// second one wants.  K pages are [page, kv_head, offset, head_dim] and V pages
// [page, kv_head, head_dim, offset]: in both, the contraction index of the
// product they feed is contiguous, so every operand is loaded from memory
// straight into registers, with no staging in LDS and no barrier in the loop.
// Heads that share a KV head share every K and V register: a step computes
// all their scores first, then walks V once.  Comparisons with the mask are
// made only in steps that touch the diagonal, a window's edge or the end, and
// an output is rescaled only in steps where a running maximum moved.
//
// Operand layout of v_mfma_f32_16x16x32_bf16 (lane l, g = l / 16, r = l % 16):
//   A[16 x 32]: row r,    columns 8g .. 8g+7        B[32 x 16]: column r, rows 8g .. 8g+7
//   C[16 x 16]: column r, rows 4g .. 4g+3
// A step takes 32 keys as two score tiles.  Which key a tile's row stands for is
// free, and is chosen so that lane group g ends up with the scores of the eight
// consecutive keys 8g .. 8g+7: row 4a + i of tile t is key 8a + 4t + i.  Packed
// in that order they are the B operand of O^T = V^T P^T, whose A operand is then
// eight consecutive keys of one head_dim row of V^T: one 16-byte load.
//
// Reference counterparts: the FA4 / FlashInfer paged kernels the reference
// calls (crates/prelude-cuda/src/attn/flash_v4.rs:125-277,
// crates/prelude-cuda/src/attn/flashinfer.rs:737-797); formula as in
// crates/prelude-core/src/ops/traits/attention.rs:10-99.
#include "common.h"
#include "api.h"
#include "attention_mfma_core.h"

#include <stdlib.h>

namespace pa {

// ---------------------------------------------------------------------------
// decode: grid (nkv * qtiles, splits, sequences), WAVES wavefronts (4, or 2 for small grids), each taking every
// WAVES-th step of 32 keys
// ---------------------------------------------------------------------------

// What the decode kernel needs to take the merged QKV projection as it leaves the product instead of queries
// that have been through the QK-norm + RoPE kernel: it norms and rotates its own queries, and the workgroup
// whose split holds the token's own position first norms, rotates and writes the token's key and copies its
// value into the cache (the kernel of qknorm_rope.hip, for one token and KV head).
struct FusedQkv {
  const bf16* qkv;          // [tokens, (nh + 2 nkv) * head_dim]
  const float* q_weight;    // may be null: no norm
  const float* k_weight;
  const float* cos_table;   // [positions, head_dim / 2]
  const float* sin_table;
  const int* slots;
  float eps;
};

// The sum of squares of a query's row as every decode kernel forms it, so that a query is the same bits in all of them: lane group g
// adds the elements 32 ks + 8 g .. + 7 in their order, then the four groups' sums are added.
template <int HD>
__device__ __forceinline__ float query_squares(const bf16x8 (&raw)[HD / 32]) {
  float ss = 0.f;
#pragma unroll
  for (int ks = 0; ks < HD / 32; ++ks)
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += (float)raw[ks][j] * (float)raw[ks][j];
  return xor_sum16_32(ss);
}

// One head's row of the projection normed and rotated by a wavefront: load() asks for everything at once.
template <int HD>
struct HeadRow {
  static constexpr int EPL = HD / kWave;   // 64 -> 1, 128 -> 2: a lane's elements; its rotation partner is lane ^ 32
  typedef bf16 vec_t __attribute__((ext_vector_type(EPL)));
  typedef float fvec_t __attribute__((ext_vector_type(EPL)));
  vec_t v;
  fvec_t w, cs, sn;

  __device__ __forceinline__ void load(const FusedQkv& f, const bf16* row, const float* weight, int pos, int lane) {
    const int j0 = (lane % 32) * EPL;
    v = *reinterpret_cast<const vec_t*>(row + lane * EPL);
    w = *reinterpret_cast<const fvec_t*>(weight ? weight + lane * EPL : f.cos_table + j0);   // not used without a scale
    cs = *reinterpret_cast<const fvec_t*>(f.cos_table + (size_t)pos * (HD / 2) + j0);
    sn = *reinterpret_cast<const fvec_t*>(f.sin_table + (size_t)pos * (HD / 2) + j0);
  }
  // The sum of squares of a key's row.
  __device__ __forceinline__ float squares() const {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) ss += (float)v[e] * (float)v[e];
    return wave_sum(ss);
  }
  __device__ __forceinline__ vec_t turned(const FusedQkv& f, bool scaled, int lane, float ss) const {
    float x[EPL];
    const float inv = rsqrtf(ss / (float)HD + f.eps);
    vec_t out;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      x[e] = (float)v[e];
      if (scaled) x[e] = x[e] * inv * w[e];
      const unsigned u = __float_as_uint(x[e]);
      const auto both = __builtin_amdgcn_permlane32_swap(u, u, false, false);   // [0]: the lower half's, [1]: the upper's
      const float partner = __uint_as_float(lane < 32 ? both[1] : both[0]);
      out[e] = (bf16)(lane < 32 ? x[e] * cs[e] - partner * sn[e] : partner * sn[e] + x[e] * cs[e]);
    }
    return out;
  }
};

// A token's new key and value for one KV head, a wavefront's work, stored at `slot`.
template <int HD>
__device__ __forceinline__ void store_kv(bf16* kc, bf16* vc, int slot, int nkv, int kvh, int page_shift, int lane,
                                         typename HeadRow<HD>::vec_t key, typename HeadRow<HD>::vec_t value) {
  constexpr int EPL = HeadRow<HD>::EPL;
  const int page = slot >> page_shift, off = slot & ((1 << page_shift) - 1);
  bf16* vdst = vc + ((((size_t)page * nkv + kvh) * HD) << page_shift) + off;
#pragma unroll
  for (int e = 0; e < EPL; ++e) vdst[(size_t)(lane * EPL + e) << page_shift] = value[e];
  *reinterpret_cast<typename HeadRow<HD>::vec_t*>(kc + ((((size_t)page * nkv + kvh) << page_shift) + off) * HD + lane * EPL) = key;
}

// Element i of a float4 (i known when the loops around it are unrolled).
__device__ __forceinline__ float f4(const float4& v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w)); }

// Q^T of one head as B operands from the raw projection: normed and rotated in the lane.  Lane (g, r) holds
// head_dim 32 ks + 8g .. + 7 of its head; the element head_dim / 2 further on, its rotation partner, is in
// the same lane (ks + KS / 2), and the sum of squares runs over the lane's elements and the four lane groups.
template <int HD>
__device__ __forceinline__ void fused_load_q(const FusedQkv& f, const bf16* qrow, bool valid, int pos, int g, bf16x8* qf) {
  constexpr int KS = HD / 32;
  static_assert(HD == 64 || HD == 128, "the rotation partner must sit in the same lane");
  // Everything the lane needs is asked for at once, in 16-byte pieces: its elements of the row, and for each of
  // its KS / 2 first-half stretches of eight elements the two stretches of the norm's scale and the angles' cosines
  // and sines.  (Element by element, under the test for a scale, the loads had been issued and waited for one
  // pair at a time: sixteen trips to the cache in a row.)
  bf16x8 raw[KS];
  float4 wa[KS / 2][2], wb[KS / 2][2], cs4[KS / 2][2], sn4[KS / 2][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    raw[ks] = zero8();
    if (valid) raw[ks] = *reinterpret_cast<const bf16x8*>(qrow + 32 * ks + 8 * g);
  }
#pragma unroll
  for (int ks = 0; ks < KS / 2; ++ks) {
    const int d = 32 * ks + 8 * g;   // the first-half element; its partner is d + HD / 2
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (f.q_weight) {
        wa[ks][h] = *reinterpret_cast<const float4*>(f.q_weight + d + 4 * h);
        wb[ks][h] = *reinterpret_cast<const float4*>(f.q_weight + d + HD / 2 + 4 * h);
      }
      cs4[ks][h] = *reinterpret_cast<const float4*>(f.cos_table + (size_t)pos * (HD / 2) + d + 4 * h);
      sn4[ks][h] = *reinterpret_cast<const float4*>(f.sin_table + (size_t)pos * (HD / 2) + d + 4 * h);
    }
  }
  const float inv = rsqrtf(query_squares<HD>(raw) / (float)HD + f.eps);
#pragma unroll
  for (int ks = 0; ks < KS / 2; ++ks) {
    bf16x8 lo, hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float a = (float)raw[ks][j], b = (float)raw[ks + KS / 2][j];
      if (f.q_weight) {
        a = a * inv * f4(wa[ks][j / 4], j % 4);
        b = b * inv * f4(wb[ks][j / 4], j % 4);
      }
      const float cs = f4(cs4[ks][j / 4], j % 4), sn = f4(sn4[ks][j / 4], j % 4);
      lo[j] = (bf16)(a * cs - b * sn);
      hi[j] = (bf16)(a * sn + b * cs);
    }
    qf[ks] = lo;
    qf[ks + KS / 2] = hi;
  }
}

// What attn_decode_few_kernel takes of the raw projection: a head's query a wavefront, the KV head's new key and value.
template <int HD, bool FUSED> struct FewRows {};
template <int HD> struct FewRows<HD, true> {
  HeadRow<HD> query, key;
  bf16x8 raw[HD / 32];   // the query's row as query_squares wants it
  typename HeadRow<HD>::vec_t value;
  int slot;
};
// Rows padded so that eight of them do not begin in the same bank.
template <int HD> struct FewLds {
  __align__(16) float o[8][8][HD + 4];   // [wavefront][head of the group]
  f32x2 ml[8][8];
  __align__(16) bf16 q[8][HD + 8];
  __align__(16) bf16 kv[2][HD];
};

// What the grid's layers from `nseq` on do.  A kernel without such layers is another one: with the arguments and the branch, and
// nothing to read, it took 0.15 to 0.4 us longer (32 heads over 8, 1,500 keys 10.6 against 10.2 us).
template <bool READS>
struct ReadsAhead {};
template <>
struct ReadsAhead<true> {
  int nseq;
  Ahead ahead;
};

// The splits that the sequences of a step have between them, one sequence's behind the other's: which one is the item-th, and how many
// there are (256 sequences at most, a lane each).
constexpr int kListedMost = 256;
struct Listed {
  int place, split, seq, ctx, token, total;   // place: the sequence's in the list
};
__device__ __forceinline__ int wave_running_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // one, two, four and eight lanes back in rows of sixteen,
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // the last of a row to the next one, of two to the next two
  return v + __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
}
template <typename ItemOf>
__device__ __forceinline__ Listed listed_split(const int* __restrict__ seq_ids, const int* __restrict__ cu_q,
                                               const int* __restrict__ context_lens, int nseq, int window, int split_keys, ItemOf item_of) {
  const int lane = threadIdx.x % kWave;
  constexpr int kTurns = kListedMost / kWave;
  int seqs[kTurns], ctxs[kTurns], toks[kTurns], own[kTurns], upto[kTurns], total = 0;
#pragma unroll
  for (int c = 0; c < kTurns; ++c)
    if (c == 0 || c * kWave < nseq) {                               // all asked for together
      const int i = c * kWave + lane, at = i < nseq ? i : nseq - 1;
      seqs[c] = seq_ids ? seq_ids[at] : at;
      ctxs[c] = context_lens[seqs[c]], toks[c] = cu_q[seqs[c]];
    }
#pragma unroll
  for (int c = 0; c < kTurns; ++c) {
    upto[c] = total;
    if (c == 0 || c * kWave < nseq) {
      const int lo = window > 0 && ctxs[c] > window ? ctxs[c] - window : 0;
      own[c] = c * kWave + lane < nseq ? (ctxs[c] + split_keys - 1) / split_keys - lo / split_keys : 0;
      upto[c] += wave_running_sum(own[c]);
      total = __builtin_amdgcn_readlane(upto[c], kWave - 1);
    }
  }
  const int item = item_of(total);
  Listed found{0, 0, 0, 0, 0, total};
#pragma unroll
  for (int c = kTurns - 1; c >= 0; --c) {
    const unsigned long long behind = c == 0 || c * kWave < nseq ? __ballot(upto[c] > item) : 0;   // the lanes from the item's on: sums do not fall
    if (behind) {
      const int at = __builtin_ctzll(behind);
      found.place = c * kWave + at;
      found.seq = __builtin_amdgcn_readlane(seqs[c], at), found.ctx = __builtin_amdgcn_readlane(ctxs[c], at);
      found.token = __builtin_amdgcn_readlane(toks[c], at);
      found.split = item - (__builtin_amdgcn_readlane(upto[c], at) - __builtin_amdgcn_readlane(own[c], at));
    }
  }
  return found;
}

// How a grid of attn_decode_kernel is dealt out: as it stands, or the splits that there are one behind the other.
enum DecodeOrder { kAsIs, kListed };
constexpr unsigned kStretchesFrom = 512;   // listed splits of all heads, beyond which every XCD works through a stretch of them

template <int HD, bool FUSED, int WAVES>
__global__ __launch_bounds__(WAVES* kWave, 3) void attn_decode_kernel(
    const bf16* __restrict__ q, const bf16* kc, const bf16* vc,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int nh, int nkv, int page_shift, int window, ScoreMap c,
    int split_keys, int max_splits, FusedQkv fq, int order, int nseq) {
  constexpr int OT = HD / 16;
  constexpr int KS = (HD + 31) / 32;
  __shared__ float lds_o[WAVES][16][HD + 1];
  __shared__ float lds_ml[WAVES][16][2];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int group = nh / nkv;
  const int qtiles = (group + 15) / 16;
  // The KV heads run fastest over the grid: the workgroups in flight at any time then read all heads of the same
  // pages, whole stretches of memory, instead of one head's 4 KB out of every page's nkv * 4 KB (with the splits
  // fastest, long contexts of few sequences left memory channels idle: 8 x 32,768 keys took 207 us where 64 x 4,096,
  // the same bytes, took 187; now 170 and 176).  The splits run slowest, for contexts differ and a workgroup whose sequence
  // has no such split costs the chip 3 ns: the shorter sequences' come last, when there is little else to deal out.
  int split_idx, head_idx, seq_idx, seq, ctx;
  size_t token;
  if (order == kAsIs) {
    split_idx = blockIdx.z, head_idx = blockIdx.x, seq_idx = blockIdx.y;
    seq = seq_ids ? seq_ids[seq_idx] : seq_idx;   // no list: every sequence of the step
    ctx = context_lens[seq], token = cu_q[seq];
  } else {
    const unsigned hq = nkv * qtiles;
    unsigned v = blockIdx.x;
    const Listed found = listed_split(seq_ids, cu_q, context_lens, nseq, window, split_keys, [&](int splits) {
      const unsigned total = splits * hq;
      if (total > kStretchesFrom && v < total) {
        const unsigned per = total / 8, rem = total % 8, x = v % 8;
        v = x * per + (x < rem ? x : rem) + v / 8;
      }
      return (int)(v / hq);
    });
    if (blockIdx.x >= found.total * hq) return;
    head_idx = v % hq, seq_idx = found.place, split_idx = found.split, seq = found.seq, ctx = found.ctx, token = found.token;
  }
  const int kvh = head_idx / qtiles, qt = head_idx % qtiles;
  const int pos = ctx - 1;
  const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  const int first_split = lo / split_keys;
  const int nsplit = (ctx + split_keys - 1) / split_keys - first_split;
  if (split_idx >= nsplit) return;
  const int sp = first_split + split_idx;
  const int k_begin = sp * split_keys > lo ? sp * split_keys : lo;
  const int k_end = (sp + 1) * split_keys < ctx ? (sp + 1) * split_keys : ctx;

  KeyWalk w{kc, vc, block_table + (size_t)seq * table_stride, nkv, kvh, page_shift, (1 << page_shift) - 1, lo, ctx};
  const int head = kvh * group + qt * 16 + r;  // this lane's query head
  const bool qvalid = qt * 16 + r < group;
  bf16x8 qf[1][KS];
  if constexpr (FUSED) {
    const int heads = nh + 2 * nkv;
    // a sequence that feeds one token feeds the one at its last position: no need to wait for positions[token]
    fused_load_q<HD>(fq, fq.qkv + (token * heads + (qvalid ? head : 0)) * HD, qvalid, pos, g, qf[0]);
    if (split_idx == nsplit - 1) {   // the split that holds the token's own position: its key and value first
      const int slot = fq.slots[token];
      if (wave == 0 && slot >= 0) {
        HeadRow<HD> fresh;
        fresh.load(fq, fq.qkv + (token * heads + nh + kvh) * HD, fq.k_weight, pos, lane);
        const auto value = *reinterpret_cast<const typename HeadRow<HD>::vec_t*>(fq.qkv + (token * heads + nh + nkv + kvh) * HD + lane * HeadRow<HD>::EPL);
        store_kv<HD>(const_cast<bf16*>(kc), const_cast<bf16*>(vc), slot, nkv, kvh, page_shift, lane, fresh.turned(fq, fq.k_weight != nullptr, lane, fresh.squares()), value);
      }
      __syncthreads();   // the other wavefronts read them from the cache below
    }
  } else {
    load_q<HD>(q + (token * nh + (qvalid ? head : 0)) * HD, qvalid, g, qf[0]);
  }

  HeadState<HD> st[1];
  const int step0 = (sp * split_keys) / 32;  // splits start at multiples of 32 keys
  const int steps = split_keys / 32;
  // a wavefront has two steps here (four with two wavefronts): many wavefronts per SIMD hide the latency, not a prefetch
  for (int i = wave; i < steps; i += WAVES) {
    const int key0 = (step0 + i) * 32;
    if (key0 + 32 <= k_begin || key0 >= k_end) continue;
    KFrag<HD> kf;
    load_k<HD>(w, key0, g, r, kf);
    const bool masked = key0 < k_begin || key0 + 32 > k_end;
    attend32<HD, 1>(w, key0, g, r, kf, qf, c, masked, st, [&](int key) { return key >= k_begin && key < k_end; });
  }
  // merge the wavefronts through LDS; maxima leave in the log2 domain (raw maximum times c)
  const float l_wave = st[0].l[0];
  if (g == 0) {
    lds_ml[wave][r][0] = st[0].reference();
    lds_ml[wave][r][1] = l_wave;
  }
#pragma unroll
  for (int t = 0; t < OT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_o[wave][r][16 * t + 4 * g + i] = st[0].o[t][i];
  __syncthreads();
  const int nq = group - qt * 16 < 16 ? group - qt * 16 : 16;
  for (int e = threadIdx.x; e < nq * HD; e += blockDim.x) {
    const int qi = e / HD, d = e % HD;
    float mm = lds_ml[0][qi][0];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) mm = fmaxf(mm, lds_ml[v][qi][0]);
    float o = 0.f, l = 0.f;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
      const float f = lds_ml[v][qi][0] == -INFINITY ? 0.f : exp2f(lds_ml[v][qi][0] - mm);
      o += lds_o[v][qi][d] * f;
      l += lds_ml[v][qi][1] * f;
    }
    const int h = kvh * group + qt * 16 + qi;
    if (nsplit == 1) {
      out[(token * nh + h) * HD + d] = (bf16)(o / (l + c.sink_term(h, mm)));
    } else {
      const size_t slot = ((size_t)seq_idx * nh + h) * max_splits + split_idx;
      part_o[slot * HD + d] = o;
      if (d == 0) {
        part_ml[slot * 2] = mm;
        part_ml[slot * 2 + 1] = l;
      }
    }
  }
}

// The same for grids of up to 192 workgroups (groups of up to eight heads, splits of 256 keys): eight wavefronts, a step of 32 keys
// each.  Such a grid leaves most of the chip idle, and what it takes is the longest path through one wavefront: its trips to memory, and
// its instructions at 2 to 3 ns each.  So there are two trips, lengths and page numbers (of pages that the sequence may not have: looked
// at when the length is there), then keys, values and the raw projection; a wavefront norms and turns one head's row, two elements a
// lane, and the queries, the token's own key and its value go to the others through LDS (their way to the cache is waited for by
// nobody); and a step that is a wavefront's only one rescales nothing.
// Alone in a graph, caches in the L2, in us (five trips, all rows' queries turned by every wavefront in between / this): 16 heads over
// 8 of 128, a context of 150 6.7 / 5.5, four 6.7 / 5.6, sixteen of 250 7.6 / 6.1; 32 over 8, 1,003 keys and the merge 11.0 / 9.1, 4,096
// 11.1 / 9.3.  0.17 of that is the order of query_squares: two elements a lane and a sum over the wavefront are shorter, but round some
// queries to another bfloat16 than the kernels of larger grids do.
constexpr int kFewSplit = 256;

// Eight elements with those that `which` names replaced by the halves of `bits`.
template <typename Which>
__device__ __forceinline__ bf16x8 put_bits(bf16x8 v, unsigned bits, Which which) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  u32x4 u = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned m = (which(2 * j) ? 0xffffu : 0u) | (which(2 * j + 1) ? 0xffff0000u : 0u);
    u[j] = (u[j] & ~m) | (bits & m);
  }
  return __builtin_bit_cast(bf16x8, u);
}

// FOUR: pages of four keys, so that a lane's eight keys of V, and its rows of the two tiles of K, lie in two pages (16 heads over 8,
// four contexts of 150, 6.0 us where attn_decode_kernel with its four wavefronts takes 6.8; 32 over 8, 1,003 keys 9.6 and 11.0).
template <int HD, bool FUSED, bool READS, bool FOUR>
__global__ __launch_bounds__(8 * kWave, 1) void attn_decode_few_kernel(
    const bf16* __restrict__ q, const bf16* kc, const bf16* vc,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int nh, int nkv, int page_shift, int window, ScoreMap c,
    int max_splits, FusedQkv fq, ReadsAhead<READS> also) {
  constexpr int OT = HD / 16, KS = (HD + 31) / 32;
  constexpr int P = FOUR ? 2 : 1, kRun = 8 / P;   // pages of a lane's eight keys, and neighbouring keys of one
  __shared__ FewLds<HD> lds;
  if constexpr (READS) {
    if (blockIdx.z >= (unsigned)also.nseq) {
      const int first = gridDim.x * gridDim.y * also.nseq;
      const int flat = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
      read_ahead(also.ahead, flat - (first + 7) / 8 * 8, 8 * kWave);
      return;
    }
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int group = nh / nkv, kvh = blockIdx.x, split_idx = blockIdx.y, seq_idx = blockIdx.z;
  const int seq = seq_ids ? seq_ids[seq_idx] : seq_idx;
  const int* table = block_table + (size_t)seq * table_stride;
  const int ctx = context_lens[seq];
  const size_t token = cu_q[seq];
  int lo = 0;
  if (window > 0) {
    lo = ctx - window > 0 ? ctx - window : 0;
    asm volatile("" ::: "memory");   // a branch: without a window nothing up to the page numbers waits for the length
  }
  const int sp = lo / kFewSplit + split_idx, key0 = sp * kFewSplit + wave * 32;
  const int page_mask = (1 << page_shift) - 1;
  // pages of the lane's eight keys of K (rows of both tiles) and of V, and of the step's first visible key, which stands in for
  // keys that are not seen; entries behind the table's width are not asked for
  const int kb = key0 + 8 * (r / 4), vb = key0 + 8 * g, fk = key0 > lo ? key0 : lo;
  auto entry = [&](int key) {
    const int at = (key > lo ? key : lo) >> page_shift;
    // (a relaxed load of this wavefront's: an ordinary one is moved behind the test for the split)
    return __hip_atomic_load(table + (at < table_stride ? at : table_stride - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  int kpage[P], vpage[P];
#pragma unroll
  for (int i = 0; i < P; ++i) kpage[i] = entry(kb + kRun * i), vpage[i] = entry(vb + kRun * i);
  const int fpage = entry(fk);
  const int pos = ctx - 1;
  const int nsplit = (ctx + kFewSplit - 1) / kFewSplit - lo / kFewSplit;
  if (split_idx >= nsplit) return;
  const bool active = key0 + 32 > lo && key0 < ctx;
  const int heads = nh + 2 * nkv;

  bf16x8 qf[KS];
  FewRows<HD, FUSED> rows;
  const bool last = split_idx == nsplit - 1;   // holds the token's own position
  if constexpr (FUSED) {
    rows.slot = fq.slots[token];
    const bf16* kv = fq.qkv + (token * heads + nh + kvh) * HD;
    const bf16* qrow = fq.qkv + (token * heads + kvh * group + (wave < group ? wave : 0)) * HD;
    rows.query.load(fq, qrow, fq.q_weight, pos, lane);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rows.raw[ks] = *reinterpret_cast<const bf16x8*>(qrow + 32 * ks + 8 * g);
    rows.key.load(fq, kv, fq.k_weight, pos, lane);
    rows.value = *reinterpret_cast<const typename HeadRow<HD>::vec_t*>(kv + nkv * HD + lane * HeadRow<HD>::EPL);
  } else {
    load_q<HD>(q + (token * nh + kvh * group + (r < group ? r : 0)) * HD, true, g, qf);
  }
  KFrag<HD> kf;
  // where in the pool, in keys; a wavefront without keys brings the pool's first ones, and a key that is not seen fk's
  int krow[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int key = kb + 4 * t + r % 4;
    const bool in = key >= lo && key < ctx;
    krow[t] = active ? ((in ? kpage[t % P] : fpage) << page_shift) + ((in ? key : fk) & page_mask) : 0;
    const size_t row = (((size_t)(krow[t] >> page_shift) * nkv + kvh) << page_shift) + (krow[t] & page_mask);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      kf.k[t][s] = zero8();
      if (HD % 32 == 0 || 32 * s + 8 * g < HD) kf.k[t][s] = *reinterpret_cast<const bf16x8*>(kc + row * HD + 32 * s + 8 * g);
    }
  }
  int vrow[P];
  typedef bf16 run_t __attribute__((ext_vector_type(kRun)));
  run_t vruns[P][OT];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int key = vb + kRun * i;
    const bool in = key + kRun > lo && key < ctx;
    vrow[i] = active ? ((in ? vpage[i] : fpage) << page_shift) + ((in ? key : fk & ~(kRun - 1)) & page_mask) : 0;
    const bf16* vp = vc + ((((size_t)(vrow[i] >> page_shift) * nkv + kvh) * HD) << page_shift) + (vrow[i] & page_mask);
#pragma unroll
    for (int t = 0; t < OT; ++t) vruns[i][t] = *reinterpret_cast<const run_t*>(vp + ((size_t)(16 * t + r) << page_shift));
  }
  __builtin_amdgcn_sched_barrier(0);   // all of it on its way before anything is waited for
  bf16x8 va[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    if constexpr (FOUR) va[t] = __builtin_shufflevector(vruns[0][t], vruns[1][t], 0, 1, 2, 3, 4, 5, 6, 7);
    else va[t] = vruns[0][t];
  }
  if constexpr (FUSED) {
    typedef typename HeadRow<HD>::vec_t vec_t;
    constexpr int EPL = HeadRow<HD>::EPL;
    if (wave < group)
      *reinterpret_cast<vec_t*>(&lds.q[wave][lane * EPL]) = rows.query.turned(fq, fq.q_weight != nullptr, lane, query_squares<HD>(rows.raw));
    const bool fresh = last && rows.slot >= 0;   // the same in all wavefronts
    if (fresh && wave == 7) {
      const vec_t key = rows.key.turned(fq, fq.k_weight != nullptr, lane, rows.key.squares());
      *reinterpret_cast<vec_t*>(&lds.kv[0][lane * EPL]) = key;
      *reinterpret_cast<vec_t*>(&lds.kv[1][lane * EPL]) = rows.value;
      store_kv<HD>(const_cast<bf16*>(kc), const_cast<bf16*>(vc), rows.slot, nkv, kvh, page_shift, lane, key, rows.value);
    }
    asm volatile("s_waitcnt lgkmcnt(0)\ns_barrier" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(&lds.q[r < group ? r : 0][32 * ks + 8 * g]);
    if (fresh && active) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (krow[t] == rows.slot) {
#pragma unroll
          for (int s = 0; s < KS; ++s) kf.k[t][s] = *reinterpret_cast<const bf16x8*>(&lds.kv[0][32 * s + 8 * g]);
        }
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int at = rows.slot - vrow[i];
        if (at >= 0 && at < kRun) {
#pragma unroll
          for (int t = 0; t < OT; ++t) {
            const unsigned v = *reinterpret_cast<const unsigned short*>(&lds.kv[1][16 * t + r]) * 0x10001u;
            va[t] = put_bits(va[t], v, [&](int e) { return e == kRun * i + at; });
          }
        }
      }
    }
  }
  // attend32_core with sums that are still zero
  f32x4 l{0.f, 0.f, 0.f, 0.f}, o[OT];
  float reference = -INFINITY;   // log2 domain: the largest raw score times c
#pragma unroll
  for (int t = 0; t < OT; ++t) o[t] = l;
  if (active) {
    const bool masked = key0 < lo || key0 + 32 > ctx;
    if (masked) {                      // what lies beside the keys may be anything
#pragma unroll
      for (int t = 0; t < OT; ++t) va[t] = put_bits(va[t], 0u, [&](int e) { return vb + e < lo || vb + e >= ctx; });
    }
    float s[8];
    const float mx = xor_max16_32(scores32<HD>(key0, g, kf, qf, masked, c, s, [&](int key) { return key >= lo && key < ctx; }));
    float shift = 0.f;
    if (mx > -INFINITY) {
      shift = -mx * c.c;
      reference = -shift;
    }
    const bf16x8 pb = probabilities(s, c.c, shift);
    l = mfma16(ones8(), pb, l);
#pragma unroll
    for (int t = 0; t < OT; ++t) o[t] = mfma16(va[t], pb, o[t]);
  }
  // the wavefronts' sums through LDS, in their order
  if (r < group) {
    if (g == 0) lds.ml[wave][r] = f32x2{reference, l[0]};
#pragma unroll
    for (int t = 0; t < OT; ++t) *reinterpret_cast<f32x4*>(&lds.o[wave][r][16 * t + 4 * g]) = o[t];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < group * HD; e += 8 * kWave) {
    const int qi = e / HD, d = e % HD, h = kvh * group + qi;
    f32x2 ml[8];
    float part[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) ml[v] = lds.ml[v][qi], part[v] = lds.o[v][qi][d];
    float mm = ml[0][0];
#pragma unroll
    for (int v = 1; v < 8; ++v) mm = fmaxf(mm, ml[v][0]);
    float sum = 0.f, lsum = 0.f;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const float f = ml[v][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[v][0] - mm);
      sum += part[v] * f;
      lsum += ml[v][1] * f;
    }
    if (nsplit == 1) {
      out[(token * nh + h) * HD + d] = (bf16)(sum / (lsum + c.sink_term(h, mm)));
    } else {
      const size_t slot = ((size_t)seq_idx * nh + h) * max_splits + split_idx;
      part_o[slot * HD + d] = sum;
      if (d == 0) *reinterpret_cast<f32x2*>(part_ml + slot * 2) = f32x2{mm, lsum};
    }
  }
}

// Merges the splits of one (sequence, head): grid (nh, sequences), groups of a thread per head_dim column.
// Every wavefront keeps a split per lane (maximum, weight), sixteen splits' outputs are asked for before the
// weights are known, and the sums run over the splits in order.  The splits go to the groups in runs of 64
// (run c to group c mod merge_groups_of(HD)), and the groups' sums are added in group order: a request's result
// depends on its own number of splits alone, and up to 64 splits (16,384 keys) it is one group's sum as it
// stands.  The launch brings as many groups as the longest context has runs (eight at most): a merge of 512
// splits by one group waits 32 times for memory, one after the other.
constexpr int kMergeGroups = 8;
constexpr long kMergeFew = 1024;   // workgroups
// ... as far as a workgroup's 1,024 threads go: heads wider than 128 get fewer groups
constexpr int merge_groups_of(int hd) {
  const int threads = (hd + kWave - 1) / kWave * kWave;
  return kMergeGroups * threads <= 1024 ? kMergeGroups : 1024 / threads;
}

template <int HD, bool FEW>
__global__ __launch_bounds__(merge_groups_of(HD) * ((HD + kWave - 1) / kWave * kWave)) void attn_decode_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out, int nh, int window,
    int split_keys, int max_splits, const float* __restrict__ sink) {
  constexpr int kBatch = 16;
  constexpr int TPG = (HD + kWave - 1) / kWave * kWave;   // threads a group
  __shared__ float group_acc[kMergeGroups][TPG];
  __shared__ float group_l[kMergeGroups];
  const int h = blockIdx.x;
  const int groups = blockDim.x / TPG;                     // the launch's: all runs of the longest context, or eight
  const int grp = threadIdx.x / TPG, d = threadIdx.x % TPG, lane = threadIdx.x % kWave;
  const bool col = d < HD;
  const size_t base = ((size_t)blockIdx.y * nh + h) * max_splits;
  const float* po = part_o + base * HD + (col ? d : 0);
  const int first = grp * kWave;                           // this group's first run
  const int seq = seq_ids ? seq_ids[blockIdx.y] : (int)blockIdx.y;
  const int ctx = context_lens[seq];
  const size_t token = cu_q[seq];
  const int pos = ctx - 1;
  const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  const int nsplit = (ctx + split_keys - 1) / split_keys - lo / split_keys;
  // the first batch of outputs and a lane's first split, on their way while the weights are worked out, and of FEW workgroups while the
  // length comes: of splits that the context may not have (with attention, us, before / now: 3 x 1,003 keys 9.4 / 8.8, 8 x 4,097
  // 29.0 / 28.0; 48 of 61 to 4,096, 1,536 workgroups, 42.7 / 43.3 without the limit)
  float o[kBatch];
  f32x2 own;
  const auto ask = [&](int most) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) o[i] = po[(size_t)min(first + i, most - 1) * HD];
    own = *reinterpret_cast<const f32x2*>(part_ml + (base + min(lane, most - 1)) * 2);
  };
  if constexpr (FEW) {
    ask(max_splits);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (nsplit <= 1) return;  // written by the first kernel
  if constexpr (!FEW) ask(nsplit);
  float mm = lane < nsplit ? own[0] : -INFINITY;
  for (int s = lane + kWave; s < nsplit; s += kWave) mm = fmaxf(mm, part_ml[(base + s) * 2]);
  mm = wave_max(mm);
  float acc = 0.f, l = 0.f;
  for (int s0 = first; s0 < nsplit; s0 += merge_groups_of(HD) * kWave) {   // a split per lane; in order of the splits
    const int s = s0 + lane;
    float f = 0.f, ls = 0.f;
    if (s < nsplit) {
      const f32x2 ml = s < kWave ? own : *reinterpret_cast<const f32x2*>(part_ml + (base + s) * 2);
      f = exp2f(ml[0] - mm);
      ls = ml[1] * f;
    }
    l += wave_sum(ls);
    const int count = nsplit - s0 < kWave ? nsplit - s0 : kWave;
    for (int b0 = 0; b0 < count; b0 += kBatch) {
      if (s0 + b0 > first) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) o[i] = (col && b0 + i < count) ? po[(size_t)(s0 + b0 + i) * HD] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        // the index is the same in every lane: a read of one lane's register, no exchange
        const float fi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), b0 + i < kWave ? b0 + i : 0));
        if (b0 + i < count) acc += o[i] * fi;
      }
    }
  }
  // a sink joins the finished sums once, against the same maximum as the splits
  const float sink_l = sink ? exp2f(sink[h] * kLog2e - mm) : 0.f;
  if (groups == 1) {
    if (col) out[(token * nh + h) * HD + d] = (bf16)(acc / (l + sink_l));
    return;
  }
  group_acc[grp][d] = acc;
  if (d == 0) group_l[grp] = l;
  __syncthreads();
  if (grp == 0 && col) {
    float a = group_acc[0][d], ll = group_l[0];
    for (int g = 1; g < groups; ++g) {
      a += group_acc[g][d];
      ll += group_l[g];
    }
    out[(token * nh + h) * HD + d] = (bf16)(a / (ll + sink_l));
  }
}

// ---------------------------------------------------------------------------
// prefill: grid (pairs of 64-token tiles, nkv * head groups, sequences); a wavefront owns 16 tokens x GT heads
// ---------------------------------------------------------------------------
// One wavefront's share of a 64-token tile: 16 tokens from t0, all keys they may see.
template <int HD, int GT>
__device__ __forceinline__ void prefill_tile(const bf16* __restrict__ q, bf16* __restrict__ out, const bf16* kc,
                                             const bf16* vc, const int* table, int row0, int q_len, int ctx, int t0,
                                             int nh, int nkv, int kvh, int head0, int page_shift, int window,
                                             const ScoreMap& c, int g, int r) {
  constexpr int OT = HD / 16;
  constexpr int KS = (HD + 31) / 32;
  const int start = ctx - q_len;                // position of the portion's first token
  const bool qvalid = t0 + r < q_len;
  const int my_pos = start + t0 + r;            // this lane's query position
  const int last_valid = t0 + 15 < q_len ? t0 + 15 : q_len - 1;
  const int last_pos = start + last_valid;
  const int first_pos = start + t0;
  const int lo = (window > 0 && first_pos - window + 1 > 0) ? first_pos - window + 1 : 0;
  const int hi = last_pos + 1;
  const int my_lo = (window > 0 && my_pos - window + 1 > 0) ? my_pos - window + 1 : 0;
  // keys every valid query of the tile sees: from the last token's window start up to the first token's position
  const int all_lo = (window > 0 && last_pos - window + 1 > 0) ? last_pos - window + 1 : 0;
  const int all_hi = first_pos + 1;

  KeyWalk w{kc, vc, table, nkv, kvh, page_shift, (1 << page_shift) - 1, lo, hi};
  bf16x8 qf[GT][KS];
  HeadState<HD> st[GT];
#pragma unroll
  for (int j = 0; j < GT; ++j)
    load_q<HD>(q + ((size_t)(row0 + (qvalid ? t0 + r : 0)) * nh + head0 + j) * HD, qvalid, g, qf[j]);

  int key0 = (lo / 32) * 32;
  KFrag<HD> kf_next;
  load_k<HD>(w, key0, g, r, kf_next);
  for (; key0 < hi; key0 += 32) {
    const KFrag<HD> kf = kf_next;
    if (key0 + 32 < hi) load_k<HD>(w, key0 + 32, g, r, kf_next);   // the next step's K rows, a step ahead
    const bool masked = key0 < all_lo || key0 + 32 > all_hi;
    attend32<HD, GT>(w, key0, g, r, kf, qf, c, masked, st, [&](int key) { return key >= my_lo && key <= my_pos; });
  }
  if (!qvalid) return;
#pragma unroll
  for (int j = 0; j < GT; ++j) {
    const float inv = 1.0f / (st[j].l[0] + c.sink_term(head0 + j, st[j].reference()));
    bf16* orow = out + ((size_t)(row0 + t0 + r) * nh + head0 + j) * HD;
#pragma unroll
    for (int t = 0; t < OT; ++t) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(st[j].o[t][i] * inv);
      *reinterpret_cast<bf16x4*>(orow + 16 * t + 4 * g) = v;
    }
  }
}

// A workgroup takes the tiles p and (last - p) of its sequence: under the causal mask a late tile sees many
// keys and an early one few, and a pair always sees about the same number, so workgroups finish together.
template <int HD, int GT>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out, int nh, int nkv,
    int page_shift, int window, ScoreMap c, int paired) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int group = nh / nkv;
  const int hgroups = group / GT;
  const int kvh = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;   // head groups fastest over the grid
  const int seq = seq_ids[blockIdx.z];
  const int row0 = cu_q[seq];
  const int q_len = cu_q[seq + 1] - row0;
  const int ctx = context_lens[seq];
  const int tiles = (q_len + 63) / 64;
  // unpaired: one tile per workgroup, late (long) tiles first
  const int first = paired ? (int)blockIdx.y : tiles - 1 - (int)blockIdx.y;
  const int second = paired ? tiles - 1 - (int)blockIdx.y : first;
  if (first > second || first < 0) return;
  const int* table = block_table + (size_t)seq * table_stride;
  const int head0 = kvh * group + hg * GT;
  {
    const int t0 = second * 64 + wave * 16;   // the long one first
    if (t0 < q_len)
      prefill_tile<HD, GT>(q, out, kc, vc, table, row0, q_len, ctx, t0, nh, nkv, kvh, head0, page_shift, window, c, g, r);
  }
  if (first != second) {
    const int t0 = first * 64 + wave * 16;
    if (t0 < q_len)
      prefill_tile<HD, GT>(q, out, kc, vc, table, row0, q_len, ctx, t0, nh, nkv, kvh, head0, page_shift, window, c, g, r);
  }
}

// ---------------------------------------------------------------------------
// prefill with the keys staged in LDS: grid as above; the four wavefronts of a workgroup own 16 tokens each
// of one 64-token tile and see almost the same keys, so the workgroup reads every block of 64 keys from the
// cache once (each thread a few 16-byte pieces, a block ahead, into registers), puts it into one of two LDS
// buffers, and all four take their MFMA operands from there.  One barrier a block.
//
// LDS layout: K rows [key][head_dim], the keys of each 32 in the order the score tiles want them (key
// 8a + 4t + i in row 16t + 4a + i); V^T rows [head_dim][64 keys], keys in their own order.  Rows are padded
// to 32 bytes past a multiple of 64: measured on gfx950, 16-byte reads of sixteen rows at such a stride run
// at the full 256 bytes a cycle, and at half that with 16 bytes of padding.
// ---------------------------------------------------------------------------
constexpr int kStageKeys = 64;

template <int HD>
struct StageLds {
  static constexpr int KROW = (2 * HD + 63) / 64 * 32 + 16;   // elements
  static constexpr int VROW = kStageKeys + 16;
  bf16 k[2][kStageKeys][KROW];
  bf16 v[2][HD][VROW];
};

// A thread's share of the staging, for workgroups of WAVES = 4 or 8 wavefronts.  Wavefront w takes the
// KW = 64 / WAVES keys KW w .. of a block of 64: of K, lane (r = lane / QL, q = lane % QL; QL = 64 / KW) takes the
// 16-byte pieces q, q + QL, .. of key KW w + r, so that the lanes of a load cover whole 64-byte stretches of a row
// (a lane per row would ask the memory pipeline for four times as many of them); of V^T, lane (d = lane / HL, h = lane % HL; HL = KW / 8 halves)
// takes the eight keys KW w + 8h .. + 7 of the rows d, d + 64 / HL, ...  Pages hold 8 keys or more here, a power of
// two: a block of 64 starts at a page's first key or lies inside one page, so a thread reads one page of each cache
// per block, `base` keys into it (always 0 for pages of up to 64 keys).  A page outside the pages [lo_page, hi_page]
// that hold the tile's keys is replaced by the nearest of those; the scores of its keys are masked.
template <int HD, int WAVES>
struct Stage {
  static_assert(WAVES == 4 || WAVES == 8, "four or eight wavefronts stage a block");
  static constexpr int KW = kStageKeys / WAVES;   // keys a wavefront stages
  static constexpr int QL = kWave / KW;           // lane groups along a K row
  static constexpr int HL = KW / 8;               // 8-key halves of a wavefront's keys
  static constexpr int DL = kWave / HL;           // V^T rows a wavefront covers at once
  static constexpr int CPK = HD / 8;              // 16-byte pieces per K row
  static constexpr int NK = (CPK + QL - 1) / QL;
  static constexpr int NV = (HD + DL - 1) / DL;
  bf16x8 k[NK];
  bf16x8 v[NV];
  int kpage, vpage, base;

  __device__ __forceinline__ void load_pages(const KeyWalk& w, int key0, int wave, int lane, int lo_page, int hi_page) {
    base = key0 & w.page_mask;
    int kp = (key0 + KW * wave + lane / QL) >> w.page_shift;
    int vp = (key0 + KW * wave + 8 * (lane % HL)) >> w.page_shift;
    kp = kp < lo_page ? lo_page : (kp > hi_page ? hi_page : kp);
    vp = vp < lo_page ? lo_page : (vp > hi_page ? hi_page : vp);
    kpage = w.table[kp];
    vpage = w.table[vp];
  }

  __device__ __forceinline__ void load(const KeyWalk& w, int wave, int lane) {
    const unsigned page_elems = ((unsigned)w.nkv * HD) << w.page_shift;   // elements per page, all KV heads
    const unsigned head_off = ((unsigned)w.kvh * HD) << w.page_shift;
    const int r = lane / QL, q = lane % QL;
    const bf16* kp = w.kc + ((unsigned long long)(unsigned)kpage * page_elems + head_off +
                             (unsigned)((base + KW * wave + r) & w.page_mask) * HD + 8 * q);
#pragma unroll
    for (int j = 0; j < NK; ++j)
      if (CPK % QL == 0 || QL * j + q < CPK) k[j] = *reinterpret_cast<const bf16x8*>(kp + 8 * QL * j);
    const int d = lane / HL, h = lane % HL;
    const bf16* vp = w.vc + ((unsigned long long)(unsigned)vpage * page_elems + head_off + ((unsigned)d << w.page_shift) +
                             (unsigned)((base + KW * wave + 8 * h) & w.page_mask));
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (HD % DL == 0 || d + DL * j < HD) v[j] = *reinterpret_cast<const bf16x8*>(vp + ((size_t)(DL * j) << w.page_shift));
  }

  __device__ __forceinline__ void store(StageLds<HD>& lds, int buf, int wave, int lane) const {
    const int r = lane / QL, q = lane % QL;
    const int key = KW * wave + r;   // 32 s + 8 a + 4 t + i  ->  row 32 s + 16 t + 4 a + i
    const int row = (key & 32) | ((key & 4) << 2) | ((key & 24) >> 1) | (key & 3);
#pragma unroll
    for (int j = 0; j < NK; ++j)
      if (CPK % QL == 0 || QL * j + q < CPK) *reinterpret_cast<bf16x8*>(&lds.k[buf][row][8 * (QL * j + q)]) = k[j];
    const int d = lane / HL, h = lane % HL;
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (HD % DL == 0 || d + DL * j < HD) *reinterpret_cast<bf16x8*>(&lds.v[buf][d + DL * j][KW * wave + 8 * h]) = v[j];
  }
};

// One step over the 32 keys `sub` of the staged block.
template <int HD, int GT, typename Visible>
__device__ __forceinline__ void attend32_lds(const StageLds<HD>& lds, int buf, int sub, int key0, int g, int r,
                                             const bf16x8 (*qf)[(HD + 31) / 32], const ScoreMap& c, bool masked,
                                             HeadState<HD>* st, Visible vis) {
  constexpr int OT = HeadState<HD>::OT;
  KFrag<HD> kf;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < KFrag<HD>::KS; ++ks) {
      if (HD % 32 == 0 || 32 * ks + 8 * g < HD) {
        kf.k[t][ks] = *reinterpret_cast<const bf16x8*>(&lds.k[buf][32 * sub + 16 * t + r][32 * ks + 8 * g]);
      } else {
        kf.k[t][ks] = zero8();
      }
    }
  bf16x8 va[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) va[t] = *reinterpret_cast<const bf16x8*>(&lds.v[buf][16 * t + r][32 * sub + 8 * g]);
  attend32_core<HD, GT>(key0, g, kf, va, qf, c, masked, st, vis);
}

// A 64-token tile from tile0 for GT * HW heads from head0: wavefront `wave` owns the tokens 16 (wave % 4) .. + 15 of
// the GT heads from head0 + GT (wave / 4).  Every wavefront takes part in the staging and the barriers, also one
// whose tokens lie beyond the portion's end.
template <int HD, int GT, int HW>
__device__ __forceinline__ void prefill_tile_lds(StageLds<HD>& lds, const bf16* __restrict__ q, bf16* __restrict__ out,
                                                 const bf16* kc, const bf16* vc, const int* table, int row0, int q_len,
                                                 int ctx, int tile0, int nh, int nkv, int kvh, int head0, int page_shift,
                                                 int window, const ScoreMap& c, int wave, int g, int r) {
  constexpr int OT = HD / 16;
  constexpr int KS = (HD + 31) / 32;
  const int lane = 16 * g + r;
  const int start = ctx - q_len;                // position of the portion's first token
  const int t0 = tile0 + 16 * (wave % 4);
  head0 += GT * (wave / 4);
  const bool wave_on = t0 < q_len;
  const bool qvalid = t0 + r < q_len;
  const int my_pos = start + t0 + r;            // this lane's query position
  const int last_valid = t0 + 15 < q_len ? t0 + 15 : q_len - 1;
  const int last_pos = start + last_valid;
  const int first_pos = start + t0;
  const int lo = (window > 0 && first_pos - window + 1 > 0) ? first_pos - window + 1 : 0;
  const int hi = last_pos + 1;
  const int my_lo = (window > 0 && my_pos - window + 1 > 0) ? my_pos - window + 1 : 0;
  const int all_lo = (window > 0 && last_pos - window + 1 > 0) ? last_pos - window + 1 : 0;
  const int all_hi = first_pos + 1;
  // what the workgroup stages: from the first token's window start to the last valid token of the tile
  const int wg_first = start + tile0;
  const int wg_last = start + (tile0 + 63 < q_len ? tile0 + 63 : q_len - 1);
  const int wg_lo = (window > 0 && wg_first - window + 1 > 0) ? wg_first - window + 1 : 0;
  const int wg_hi = wg_last + 1;

  KeyWalk w{kc, vc, table, nkv, kvh, page_shift, (1 << page_shift) - 1, wg_lo, wg_hi};
  bf16x8 qf[GT][KS];
  HeadState<HD> st[GT];
#pragma unroll
  for (int j = 0; j < GT; ++j)
    load_q<HD>(q + ((size_t)(row0 + (qvalid ? t0 + r : 0)) * nh + head0 + j) * HD, qvalid, g, qf[j]);

  Stage<HD, 4 * HW> stage;
  const int lo_page = wg_lo >> page_shift, hi_page = (wg_hi - 1) >> page_shift;
  // A block is put into LDS a whole block before it is used: while the wavefronts work on block b out of one
  // buffer, each first writes its share of block b + 1 (asked for from memory a block ago) into the other and asks
  // for block b + 2; the barrier at the block's end then says both that block b + 1 is complete and that nobody
  // reads block b any more.  (Written right before its use, the LDS writes and the barrier stood between every
  // block's arrival and its first product.)
  int key0 = (wg_lo / kStageKeys) * kStageKeys;
  stage.load_pages(w, key0, wave, lane, lo_page, hi_page);
  stage.load(w, wave, lane);
  if (key0 + kStageKeys < wg_hi) stage.load_pages(w, key0 + kStageKeys, wave, lane, lo_page, hi_page);
  stage.store(lds, 0, wave, lane);
  if (key0 + kStageKeys < wg_hi) {
    stage.load(w, wave, lane);
    if (key0 + 2 * kStageKeys < wg_hi) stage.load_pages(w, key0 + 2 * kStageKeys, wave, lane, lo_page, hi_page);
  }
  __syncthreads();
  int buf = 0;
  for (; key0 < wg_hi; key0 += kStageKeys, buf ^= 1) {
    if (key0 + kStageKeys < wg_hi) {
      stage.store(lds, buf ^ 1, wave, lane);   // the next block, asked for a block ago
      if (key0 + 2 * kStageKeys < wg_hi) {
        stage.load(w, wave, lane);             // the one after it, from the pages looked up a block ago
        if (key0 + 3 * kStageKeys < wg_hi)
          stage.load_pages(w, key0 + 3 * kStageKeys, wave, lane, lo_page, hi_page);
      }
    }
    if (wave_on) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int k32 = key0 + 32 * sub;
        if (k32 + 32 <= lo || k32 >= hi) continue;
        const bool masked = k32 < all_lo || k32 + 32 > all_hi;
        attend32_lds<HD, GT>(lds, buf, sub, k32, g, r, qf, c, masked, st,
                             [&](int key) { return key >= my_lo && key <= my_pos; });
      }
    }
    __syncthreads();
  }
  // (the loop's last barrier leaves the buffers free for the next tile)
  if (!qvalid) return;
#pragma unroll
  for (int j = 0; j < GT; ++j) {
    const float inv = 1.0f / (st[j].l[0] + c.sink_term(head0 + j, st[j].reference()));
    bf16* orow = out + ((size_t)(row0 + t0 + r) * nh + head0 + j) * HD;
#pragma unroll
    for (int t = 0; t < OT; ++t) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16)(st[j].o[t][i] * inv);
      *reinterpret_cast<bf16x4*>(orow + 16 * t + 4 * g) = v;
    }
  }
}

template <int HD, int GT, int HW>
__global__ __launch_bounds__(256 * HW, 2) void attn_prefill_lds_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_ids,
    const int* __restrict__ cu_q, const int* __restrict__ context_lens, bf16* __restrict__ out, int nh, int nkv,
    int page_shift, int window, ScoreMap c, int paired) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  StageLds<HD>& lds = *reinterpret_cast<StageLds<HD>*>(lds_raw);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int g = lane / 16, r = lane % 16;
  const int group = nh / nkv;
  const int hgroups = group / (GT * HW);
  const int kvh = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;   // head groups fastest over the grid
  // paired 2: unpaired, and the tiles (not the sequences) slowest over the grid, so that the long tiles of every
  // sequence are handed out before any short one
  const bool tile_slowest = paired == 2;
  const int seq = seq_ids[tile_slowest ? blockIdx.y : blockIdx.z];
  const int at = tile_slowest ? (int)blockIdx.z : (int)blockIdx.y;
  const int row0 = cu_q[seq];
  const int q_len = cu_q[seq + 1] - row0;
  const int ctx = context_lens[seq];
  const int tiles = (q_len + 63) / 64;
  const int first = paired == 1 ? at : tiles - 1 - at;
  const int second = paired == 1 ? tiles - 1 - at : first;
  if (first > second || first < 0) return;   // the same for the whole workgroup
  const int* table = block_table + (size_t)seq * table_stride;
  const int head0 = kvh * group + hg * GT * HW;
  prefill_tile_lds<HD, GT, HW>(lds, q, out, kc, vc, table, row0, q_len, ctx, second * 64, nh, nkv, kvh, head0,
                               page_shift, window, c, wave, g, r);   // the long one first
  if (first != second)
    prefill_tile_lds<HD, GT, HW>(lds, q, out, kc, vc, table, row0, q_len, ctx, first * 64, nh, nkv, kvh, head0,
                                 page_shift, window, c, wave, g, r);
}

// ---------------------------------------------------------------------------
// What a grid of less than one workgroup a compute unit reads ahead, in bytes: three quarters of the eight L2s of 4 MB, as
// far as the keys and values that the grid itself streams leave a window of kAheadWindow.  A decode step of (us without /
// 12 / 20 / 24 / 28 / 32 MB): 0.6B, 4 contexts of 150 893 / 863 / 845 / 836 / 830 / 833, one of 2,000 962 / 924 / 912 /
// 901 / 901 / 915, 16 of up to 250 1,121 / 1,103 / 1,078 / 1,067 / 1,083 / 1,092; 4B (whose output projection is 21 MB:
// nothing is won by a part of it), one context of 1,500 643 / 645 / 644 / 630 / 629 / 628, of 4,096 652 / 653 / 652 /
// 636 / 641 / 644; 8B (34 MB) 762 / 759 / 762 / 761 / 763 / 772.  With 25 MB of keys and values of its own (4B, 6,000
// keys) 24 MB are level and 40 MB cost 2 %.  The kernel itself takes 1.5 to 2 us longer, the products behind it 0.5 to 2.3 less
// each.  Larger grids, and the merge kernel, were no faster for reading ahead.
constexpr long long kAheadBytes = 24LL << 20;
constexpr long long kAheadWindow = 40LL << 20;

// The first units, up to `most` bytes, of a list [weights, then each one's address, bytes a unit and units].
inline Ahead ahead_cut(const long long* list, long long most, int threads) {
  Ahead a{};
  for (int i = 0; list && i < list[0] && i < kAheadMost; ++i) {
    const long long unit = list[2 + 3 * i], units = list[3 + 3 * i];
    const long long take = most / unit < units ? most / unit : units;
    if (take <= 0) break;
    a.data[i] = reinterpret_cast<const char*>(list[1 + 3 * i]);
    a.unit[i] = (int)unit, a.units[i] = (int)take;
    a.places += ahead_places((int)unit, (int)take, threads);
    if (take < units) break;
    most -= take * unit;
  }
  return a;
}

template <int HD, bool FUSED>
int launch_decode(hipStream_t st, const void* q, const void* kc, const void* vc, const int* block_table,
                  int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens, void* out,
                  float* part_o, float* part_ml, int nseq, int nh, int nkv, int page_shift, int window, float scale,
                  float softcap, const float* sink, int split_keys, int max_splits, const FusedQkv& fq,
                  const long long* ahead_list = nullptr) {
  const int qtiles = (nh / nkv + 15) / 16;
  const long total = (long)nkv * qtiles * max_splits * nseq;
  dim3 grid(nkv * qtiles, max_splits, nseq);
  // Contexts are as long as they happen to be, and the host knows the longest.  Grids of two to five rounds of the chip list the splits
  // that there are: those of a long context would come last else, with the chip all but empty.  Larger ones run on long enough,
  // and listing costs every workgroup, also those that find nothing, some 0.2 us.  With the merge, 32 heads over 8, us, before (the splits of a
  // sequence together; grids of up to 4,096 in one stretch an XCD, and so in short or long sequences) / listed / splits slowest:
  // 31 contexts of 100 to 3,000 keys 31.9 / 28.7 / 28.9, 16 of 100 to 4,000 26.0 / 21.1 / 26.7, 48 of 61 to 1,000 (16 heads over 8) 23.9 /
  // 20.0 / 21.8, of 61 to 4,096 44.4 / 41.2 / 42.4, 100 of 20 to 8,000 139 / 153 / 137, 200 of 500 to 2,000 216 / 216 / 200; with two
  // wavefronts (below) 8 of 500 to 4,096 22.7 / 18.3 / 20.6, of 4,097 29.0 / 29.5 / 29.1.  What contexts of one length lose: 20 of 3,000 44.7 /
  // 45.8 / 45.5, 4 of 32,768 115.5 / 118 / 116.5, 48 of 4,096 168 / 170 / 169.
  const int order = total > 1536 && total <= 4096 && max_splits > 1 && nseq > 1 && nseq <= kListedMost ? kListed : kAsIs;
  const dim3 dealt = order == kListed ? dim3((unsigned)total) : dim3(nkv * qtiles, nseq, max_splits);
  // Twelve wavefronts fit a compute unit (three a SIMD by their registers): three workgroups of four, 768 on the
  // chip.  A grid just above that would run a second, nearly empty round; with two wavefronts a workgroup six fit,
  // 1,536 on the chip, and the whole grid is there at once: batch 7 to 12 at 4,096 keys +0.3 to 2.3 % of the decode
  // step.  Smaller grids want the four wavefronts for their parallelism (batch 1: -3.7 % with two), larger ones
  // measured 1 to 2 % slower with two.  With two wavefronts a split's steps are added in another order (wavefront w
  // takes the steps w, w + 2, .. instead of w, w + 4, ..), so a token's sums can differ in their last bits between
  // steps whose grids fall on either side of these limits; what else is in the batch changes nothing beyond that.
  // A grid of less than one workgroup a compute unit (one sequence of 4,096 keys: 128) runs with eight, a step of
  // 32 keys each (attn_decode_few_kernel): batch 1 of a 4B model 2.518 -> 2.499 ms a step; 256 workgroups are level or better off with
  // four (13.4 against 13.7 us), and with eight up to 512 workgroups batch 3 and 4 lose 4 %.
  const bool two_wavefronts = total > 768 && total <= 1536;
  const bool eight_wavefronts = total <= 192 && nh / nkv <= 8 && split_keys == kFewSplit;
  if (eight_wavefronts) {
    const auto launch = [&](auto* kernel, auto also) {
      hipLaunchKernelGGL(kernel, grid, dim3(8 * kWave), 0, st, (const bf16*)q, (const bf16*)kc, (const bf16*)vc, block_table,
                         table_stride, seq_ids, cu_q, context_lens, (bf16*)out, part_o, part_ml, nh, nkv, page_shift, window,
                         score_map(scale, softcap, sink), max_splits, fq, also);
    };
    const long long own = total * split_keys * HD * 4, left = kAheadWindow - own;
    const Ahead ahead = ahead_cut(FUSED ? ahead_list : nullptr, left < kAheadBytes ? left : kAheadBytes, 8 * kWave);
    if constexpr (FUSED) {
      if (ahead.places) {
        // their workgroups come behind the others, from the first multiple of eight (see Ahead) in further layers of the grid
        grid.z += (unsigned)(((total + 7) / 8 * 8 - total + ahead.places + grid.x * grid.y - 1) / (grid.x * grid.y));
        if (page_shift >= 3) launch(&attn_decode_few_kernel<HD, true, true, false>, ReadsAhead<true>{nseq, ahead});
        else launch(&attn_decode_few_kernel<HD, true, true, true>, ReadsAhead<true>{nseq, ahead});
      }
    }
    if (!ahead.places) {
      if (page_shift >= 3) launch(&attn_decode_few_kernel<HD, FUSED, false, false>, ReadsAhead<false>{});
      else launch(&attn_decode_few_kernel<HD, FUSED, false, true>, ReadsAhead<false>{});
    }
  } else if (two_wavefronts) {
    hipLaunchKernelGGL((attn_decode_kernel<HD, FUSED, 2>), dealt, dim3(2 * kWave), 0, st, (const bf16*)q, (const bf16*)kc,
                       (const bf16*)vc, block_table, table_stride, seq_ids, cu_q, context_lens, (bf16*)out, part_o,
                       part_ml, nh, nkv, page_shift, window, score_map(scale, softcap, sink), split_keys, max_splits, fq, order, nseq);
  } else {
    hipLaunchKernelGGL((attn_decode_kernel<HD, FUSED, 4>), dealt, dim3(4 * kWave), 0, st, (const bf16*)q, (const bf16*)kc,
                       (const bf16*)vc, block_table, table_stride, seq_ids, cu_q, context_lens, (bf16*)out, part_o,
                       part_ml, nh, nkv, page_shift, window, score_map(scale, softcap, sink), split_keys, max_splits, fq, order, nseq);
  }
  if (int rc = check_launch("attn_decode")) return rc;
  if (max_splits > 1) {
    // a group for every run of 64 splits the longest context can have, eight at most
    const int runs = (max_splits + kWave - 1) / kWave;
    const int groups = runs < merge_groups_of(HD) ? runs : merge_groups_of(HD);
    const auto merge = [&](auto* kernel) {
      hipLaunchKernelGGL(kernel, dim3(nh, nseq), dim3(groups * ((HD + kWave - 1) / kWave * kWave)), 0, st, part_o, part_ml, seq_ids, cu_q,
                         context_lens, (bf16*)out, nh, window, split_keys, max_splits, sink);
    };
    if ((long)nh * nseq <= kMergeFew) merge(&attn_decode_merge_kernel<HD, true>);
    else merge(&attn_decode_merge_kernel<HD, false>);
    return check_launch("attn_decode_merge");
  }
  return 0;
}

template <int HD, int GT, int HW>
int launch_prefill_staged(hipStream_t st, const void* q, const void* kc, const void* vc, const int* block_table,
                          int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens, void* out,
                          int nseq, int max_q_len, int nh, int nkv, int page_shift, int window, float scale,
                          float softcap, const float* sink, int paired) {
  const int tiles = (max_q_len + 63) / 64;
  dim3 grid(nkv * (nh / nkv / (GT * HW)), paired == 1 ? (tiles + 1) / 2 : tiles, nseq);
  if (paired == 2) grid = dim3(grid.x, nseq, tiles);
  // the two buffers are more than the 64 KB a kernel may declare: asked for at launch, allowed once per kernel
  static const hipError_t allowed =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_lds_kernel<HD, GT, HW>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(StageLds<HD>));
  if (allowed != hipSuccess)
    return pa::fail("attn_prefill: %zu bytes of LDS refused: %s", sizeof(StageLds<HD>), hipGetErrorString(allowed));
  hipLaunchKernelGGL((attn_prefill_lds_kernel<HD, GT, HW>), grid, dim3(256 * HW), sizeof(StageLds<HD>), st,
                     (const bf16*)q, (const bf16*)kc, (const bf16*)vc, block_table, table_stride, seq_ids, cu_q,
                     context_lens, (bf16*)out, nh, nkv, page_shift, window, score_map(scale, softcap, sink), paired);
  return check_launch("attn_prefill");
}

template <int HD, int GT>
int launch_prefill_gt(hipStream_t st, const void* q, const void* kc, const void* vc, const int* block_table,
                      int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens, void* out,
                      int nseq, int max_q_len, int nh, int nkv, int page_shift, int window, float scale, float softcap,
                      const float* sink, int paired, int hw, bool staged) {
  const int tiles = (max_q_len + 63) / 64;
  if (!staged && paired == 2) paired = 0;   // the kernel that reads the cache itself has the one order
  dim3 grid(nkv * (nh / nkv / GT), paired == 1 ? (tiles + 1) / 2 : tiles, nseq);
  if (staged) {
    if (hw == 2)
      return launch_prefill_staged<HD, GT, 2>(st, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out,
                                              nseq, max_q_len, nh, nkv, page_shift, window, scale, softcap, sink, paired);
    return launch_prefill_staged<HD, GT, 1>(st, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out,
                                            nseq, max_q_len, nh, nkv, page_shift, window, scale, softcap, sink, paired);
  }
  hipLaunchKernelGGL((attn_prefill_kernel<HD, GT>), grid, dim3(256), 0, st, (const bf16*)q, (const bf16*)kc,
                     (const bf16*)vc, block_table, table_stride, seq_ids, cu_q, context_lens, (bf16*)out, nh, nkv,
                     page_shift, window, score_map(scale, softcap, sink), paired);
  return check_launch("attn_prefill");
}

// How a prefill launch is cut, -1 where the launcher chooses: tiles in pairs, heads a wavefront (1, 2, 4), head
// groups a workgroup (1, 2), keys staged in LDS.
struct PrefillCut {
  int paired = -1, heads = -1, groups = -1, staged = -1;
};

template <int HD>
int launch_prefill(hipStream_t st, const void* q, const void* kc, const void* vc, const int* block_table,
                   int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens, void* out, int nseq,
                   int max_q_len, int min_prefix, int nh, int nkv, int page_shift, int window, float scale,
                   float softcap, const float* sink, const PrefillCut& want) {
  const int group = nh / nkv;
  // How the work is cut: tiles in pairs (an early and a late tile of the causal triangle, so workgroups finish
  // together) and as many heads per wavefront as share the keys and fit the registers (wider heads would not fit
  // four heads' state in 256) -- unless that leaves compute units without a workgroup: a short prompt is better
  // off unpaired and with a head per wavefront.  Measured at head_dim 128: one prompt of 512 tokens takes 16 us
  // as 256 workgroups and 26 us as 64.
  // (four heads a wavefront, which heads of up to 64 wide have registers for, measured slower than two at every
  // size but 8,192 tokens, where it is level: 32 heads over 8 of 64 at 2,048 tokens 66 us against 45 and 36 with
  // two and one; the kernel stays for callers that ask for it)
  const int gt_best = group % 2 == 0 ? 2 : 1;
  const int gt_most = (HD <= 64 && group % 4 == 0) ? 4 : gt_best;   // what a caller's own cut may ask for
  const long tiles = (max_q_len + 63) / 64;
  const bool can_stage = page_shift >= 3;
  auto workgroups = [&](int p, int g_, int h_ = 1) {
    return (p ? (tiles + 1) / 2 : tiles) * nkv * (group / (g_ * h_)) * nseq;
  };
  const long enough = 256;
  int paired = tiles >= 2, gt = gt_best, hw = 1;
  // every portion has at least as many keys before it as tokens in it: its tiles see about the same number of keys
  // and need no pairing, which doubles the workgroups there are to hand out
  const bool level = min_prefix >= max_q_len;
  const bool wide_ok = can_stage && group % (gt_best * 2) == 0;   // eight wavefronts: two groups of gt_best heads
  const int gt_half = gt_best >= 2 ? gt_best / 2 : 1;
  const bool half_ok = can_stage && gt_best >= 2 && group % (gt_half * 2) == 0;
  // Pairs are workgroups of one length, so they come in rounds, and a last round that is half empty costs as much
  // as a full one: pairs pay where the rounds are full (or many).  Unpaired, the tiles are of every length from one
  // block to the whole context, the longest are handed out first, and from one and a half workgroups a compute
  // unit on they balance out by themselves.  Measured, 32 heads over 8 of 128: 1,536 tokens as 384 pairs of a head
  // a wavefront 47.2 us, unpaired with eight wavefronts 36.5; 3,072 tokens as 384 pairs 134.3, unpaired with two
  // heads a wavefront 105.0; 2,048 and 4,096 tokens, whose pairs are one full round, 53.0 and 144.5 paired against
  // 55.0 and 150.1.
  // (7,168 tokens, 448 pairs: 466 against 437 us unpaired; three prompts of 1,024, 192 pairs: 50.4 against 57.2 --
  // short tiles carry a workgroup's fixed cost less well, so one round that is three quarters full still counts)
  auto full_rounds = [&](long w, long slots) {
    return (w >= slots && (w % slots == 0 || w >= 4 * slots)) || (tiles <= 16 && 4 * w >= 3 * slots && w <= slots);
  };
  const long spread = enough * 3 / 2;
  // Two to six prompts: within a launch the workgroups are handed out sequence by sequence, so unpaired the last
  // prompt's long tiles start late; with the tiles slowest over the grid (paired 2) every prompt's long tiles
  // come first, and unpaired is ahead of pairs wherever the pairs are not exactly whole rounds (32 heads over 8 of
  // 128, us: three prompts of 512 tokens 20.0 against 22.1 in pairs and 23.2 sequence by sequence, six of 512 32.1
  // against 35.0, three of 1,024 44.6 against 49.9, three of 2,048 131.6 against 147.1; 40 heads over 8, two of 512
  // 17.7 against 23.8).  With many prompts the interleaving costs more in the L2 than the order gains (sixteen of
  // 512: 80.9 against 70.5).
  const bool few = can_stage && !level && nseq >= 2 && nseq <= 6 && tiles >= 2;
  auto whole = [&](long w, long slots) { return w >= slots && w % slots == 0; };
  if (few) {
    // the kinds of workgroup from the most heads down; of each, pairs if they are whole rounds, else unpaired if
    // there are workgroups enough to balance out
    if (wide_ok && whole(workgroups(1, gt_best, 2), enough)) {
      hw = 2;
    } else if (wide_ok && workgroups(0, gt_best, 2) >= spread) {
      paired = 2, hw = 2;
    } else if (whole(workgroups(1, gt_best, 1), 2 * enough)) {
      hw = 1;
    } else if (gt_best >= 2 && workgroups(0, gt_best, 1) >= 2 * spread) {
      paired = 2, hw = 1;
    } else if (half_ok && whole(workgroups(1, gt_half, 2), enough)) {
      gt = gt_half, hw = 2;
    } else if (half_ok && workgroups(0, gt_half, 2) >= spread) {
      paired = 2, gt = gt_half, hw = 2;
    } else {
      paired = 2, gt = gt_half, hw = 1;
    }
  } else if (wide_ok && tiles > 8 && full_rounds(workgroups(1, gt_best, 2), enough)) {
    // the most work per staged key that still gives every compute unit a workgroup (measured at head_dim 128,
    // 32 heads over 8: 4,096 tokens 171 against 186 us, 8,192 tokens 624 against 648); not for many short prompts,
    // whose workgroups are over after a few blocks (16 prompts of 512 tokens: 66 against 70 us with four
    // wavefronts a workgroup, 32 of 256: 51 against 60)
    hw = 2;
  } else if (wide_ok && tiles > 8 && !level && workgroups(0, gt_best, 2) >= spread) {
    paired = 0, hw = 2;
  } else if (level && workgroups(0, gt_best, wide_ok ? 2 : 1) >= (wide_ok ? enough : 2 * enough)) {
    // (workgroups of four wavefronts want two on a compute unit: 16 heads over 8, 2,048 tokens behind 6,144, as 256
    // of them 274 us, as 256 of eight wavefronts with a head each 166)
    paired = 0;   // 2,048 tokens behind 6,144: 297 against 342 us
    hw = wide_ok ? 2 : 1;
  } else if (level && can_stage && group % 2 == 0 && workgroups(0, 1, 2) >= enough) {
    paired = 0, gt = 1, hw = 2;   // 1,024 tokens behind 7,168: 205 against 293 us
  } else if (!wide_ok && gt_best >= 2 && tiles > 8 && full_rounds(workgroups(1, gt_best, 1), 2 * enough)) {
    // whole rounds of pairs of four wavefronts, two heads each (16 heads over 8 at 8,192 tokens: 307 against 332 us)
  } else if (half_ok && tiles > 8 && full_rounds(workgroups(1, gt_half, 2), enough)) {
    gt = gt_half, hw = 2;         // 2,048 tokens: 256 pairs of eight wavefronts, a head each
  } else if (half_ok && tiles > 8 && workgroups(0, gt_half, 2) >= spread) {
    paired = 0, gt = gt_half, hw = 2;
  } else if (half_ok && workgroups(0, gt_half, 2) == enough) {
    // exactly one workgroup of eight wavefronts a compute unit, two wavefronts a SIMD and one round (two prompts
    // of 512 tokens: 16.0 us against 17.7 as pairs of four wavefronts)
    paired = 0, gt = gt_half, hw = 2;
  } else {
    if (workgroups(paired, gt) < enough) {
      if (gt > 1 && workgroups(paired, 1) >= enough) {
        gt = 1;
      } else if (workgroups(0, gt) >= enough) {
        paired = 0;
      } else {
        paired = 0;
        gt = 1;
      }
    }
    // one workgroup per compute unit is one wavefront per SIMD, which waits for every one of its own steps: then
    // rather eight wavefronts a workgroup, half of them on the other heads (measured at 2,048 tokens: 69 against 77 us)
    // (up to one and a quarter: six prompts of 512 tokens, 384 pairs, 35.6 us as they are and 40.7 with eight wavefronts)
    if (can_stage && workgroups(paired, gt) >= enough && workgroups(paired, gt) <= enough * 5 / 4 && gt >= 2 && gt == gt_best) {
      gt /= 2;
      hw = 2;
    }
    // pairs in rounds that are not full: unpaired, if that gives workgroups enough to balance out
    // (prompts of up to 512 tokens are over too soon for rounds to form: twelve of 512 tokens 60.3 us in pairs, 64.7 without)
    if (paired && tiles > 8 && !full_rounds(workgroups(1, gt, hw), hw == 2 ? enough : 2 * enough) && workgroups(0, gt, hw) >= spread)
      paired = 0;
  }
  // keys staged in LDS for pages of 8 keys or more; pages of 4 go to the kernel that reads them itself
  bool staged = can_stage;
  // a caller's own cut (tests and measurements), where it is one the kernels have
  if (want.paired >= 0) paired = want.paired == 2 ? 2 : (want.paired != 0 && tiles >= 2);
  if (want.heads >= 0) {
    PA_REQUIRE((want.heads == 1 || want.heads == 2 || want.heads == 4) && want.heads <= gt_most,
               "attn_prefill: %d heads a wavefront, this shape takes up to %d (1, 2 or 4)", want.heads, gt_most);
    gt = want.heads;
    if (want.groups < 0) hw = 1;
  }
  if (want.groups >= 0) {
    PA_REQUIRE(want.groups == 1 || (want.groups == 2 && group % (gt * 2) == 0),
               "attn_prefill: %d head groups a workgroup with %d heads a wavefront and %d heads a KV head", want.groups,
               gt, group);
    hw = want.groups;
  }
  if (want.staged >= 0) {
    PA_REQUIRE(want.staged == 0 || staged, "attn_prefill: pages of %d keys are not staged", 1 << page_shift);
    staged = want.staged != 0;
  }
  PA_REQUIRE(staged || hw == 1, "attn_prefill: two head groups a workgroup only with staged keys");
  PA_REQUIRE(gt <= gt_most, "attn_prefill: %d heads a wavefront, head_dim %d takes up to %d", gt, HD, gt_most);
#define PA_GT(GT)                                                                                                   \
  return launch_prefill_gt<HD, GT>(st, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out, nseq, \
                                   max_q_len, nh, nkv, page_shift, window, scale, softcap, sink, paired, hw, staged)
  if constexpr (HD <= 64) {   // four heads' state of a wider head does not fit 256 registers: not built, never chosen
    if (gt == 4) PA_GT(4);
  }
  if (gt == 2) PA_GT(2);
  PA_GT(1);
#undef PA_GT
}

}  // namespace pa

using namespace pa;

#define PA_HD_SWITCH(hd, CALL)                                                                              \
  switch (hd) {                                                                                             \
    case 16: CALL(16);                                                                                      \
    case 32: CALL(32);                                                                                      \
    case 48: CALL(48);                                                                                      \
    case 64: CALL(64);                                                                                      \
    case 96: CALL(96);                                                                                      \
    case 128: CALL(128);                                                                                    \
    default: return pa::fail("MFMA attention: head_dim %d is not one of 16, 32, 48, 64, 96, 128", hd);      \
  }

static int check_common(const char* what, int nseq, int nh, int nkv, int page_size, int table_stride, int window) {
  PA_REQUIRE(nseq > 0 && nh > 0 && nkv > 0 && table_stride > 0, "%s: bad sizes sequences=%d nh=%d nkv=%d table_stride=%d",
             what, nseq, nh, nkv, table_stride);
  PA_REQUIRE(nh % nkv == 0, "%s: %d query heads are not a multiple of %d KV heads", what, nh, nkv);
  PA_REQUIRE(page_size >= 4 && (page_size & (page_size - 1)) == 0, "%s: page size %d is not a power of two >= 4", what,
             page_size);
  PA_REQUIRE(window >= 0, "%s: window %d is negative (0 means none)", what, window);
  PA_REQUIRE(nseq <= 65535, "%s: %d sequences exceed the grid", what, nseq);
  return 0;
}

// 1 if the MFMA kernels take this head_dim and page size, else 0 (the caller then uses the generic kernel).
extern "C" int pa_attn_mfma_supports(int hd, int page_size) {
  const bool hd_ok = hd == 16 || hd == 32 || hd == 48 || hd == 64 || hd == 96 || hd == 128;
  return hd_ok && page_size >= 4 && (page_size & (page_size - 1)) == 0;
}

// Workspace the decode kernel needs, in floats, for `nseq` sequences cut into at most `max_splits` splits.
extern "C" long pa_attn_decode_workspace(int nseq, int nh, int hd, int max_splits) {
  return max_splits <= 1 ? 0 : (long)nseq * nh * max_splits * (hd + 2);
}

static int attn_decode_entry(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                              int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                              void* out, float* workspace, int nseq, int nh, int nkv, int hd, int page_size,
                              int window, float scale, float softcap, const float* sink, int split_keys, int max_splits) {
  if (nseq == 0) return 0;
  PA_REQUIRE(softcap >= 0.f, "attn_decode: a score cap of %g is negative (0 means none)", (double)softcap);
  if (int rc = check_common("attn_decode", nseq, nh, nkv, page_size, table_stride, window)) return rc;
  PA_REQUIRE(split_keys >= 32 && split_keys % 32 == 0, "attn_decode: split of %d keys is not a multiple of 32", split_keys);
  PA_REQUIRE(max_splits >= 1 && max_splits <= 65535, "attn_decode: %d splits", max_splits);
  PA_REQUIRE(max_splits == 1 || workspace, "attn_decode: no workspace for %d splits", max_splits);
  float* part_o = workspace;
  float* part_ml = workspace ? workspace + (size_t)nseq * nh * max_splits * hd : nullptr;
#define PA_CALL(HD)                                                                                                  \
  return launch_decode<HD, false>((hipStream_t)stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q,         \
                                  context_lens, out, part_o, part_ml, nseq, nh, nkv, __builtin_ctz(page_size), window, \
                                  scale, softcap, sink, split_keys, max_splits, FusedQkv{})
  PA_HD_SWITCH(hd, PA_CALL)
#undef PA_CALL
}

// 1 if pa_attn_decode_fused takes these sizes: whole-width rotation of a head_dim whose half is a multiple of
// 32, and all query heads of a KV head in one tile (two workgroups must not wait for one another's key).
extern "C" int pa_attn_decode_fused_supports(int nh, int nkv, int hd, int rot, int page_size) {
  return (hd == 64 || hd == 128) && rot == hd && nkv > 0 && nh % nkv == 0 && nh / nkv <= 16 &&
         pa_attn_mfma_supports(hd, page_size);
}

// pa_qknorm_rope_kv and pa_attn_decode in one: `qkv` is the merged projection [tokens, (nh + 2 nkv) * hd] of a
// step in which the sequences `seq_ids` feed one token each; their keys and values are written to the caches
// at `slots` and their outputs to `out`; a token's position is its sequence's context length less one.  Tokens
// of other sequences are not touched.  `ahead_list` (host memory, or null): weights that the kernels behind this one stream,
// in order, [how many, then each one's address, bytes a unit and units]; a small grid reads the first of them ahead.
extern "C" int pa_attn_decode_fused(void* stream, const void* qkv, const float* q_weight, const float* k_weight,
                                    const float* cos_table, const float* sin_table, const int* slots, float eps, void* kc, void* vc, const int* block_table,
                                    int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                                    void* out, float* workspace, int nseq, int nh, int nkv, int hd, int page_size,
                                    int window, float scale, float softcap, int split_keys, int max_splits,
                                    const long long* ahead_list) {
  if (nseq == 0) return 0;
  if (ahead_list) {
    PA_REQUIRE(ahead_list[0] >= 0 && ahead_list[0] <= kAheadMost, "attn_decode_fused: %lld weights to read ahead", ahead_list[0]);
    for (int i = 0; i < ahead_list[0]; ++i) {
      const long long *w = ahead_list + 1 + 3 * i;
      PA_REQUIRE(w[0] && w[0] % 16 == 0 && w[1] >= 16 && w[1] % 16 == 0 && w[1] <= 1 << 24 && w[2] >= 1 && w[2] <= 1 << 24,
                 "attn_decode_fused: weight %d to read ahead: %lld units of %lld bytes at %#llx", i, w[2], w[1], w[0]);
    }
  }
  PA_REQUIRE(softcap >= 0.f, "attn_decode_fused: a score cap of %g is negative (0 means none)", (double)softcap);
  if (int rc = check_common("attn_decode_fused", nseq, nh, nkv, page_size, table_stride, window)) return rc;
  PA_REQUIRE(pa_attn_decode_fused_supports(nh, nkv, hd, hd, page_size), "attn_decode_fused: nh=%d nkv=%d head_dim=%d page=%d are not taken",
             nh, nkv, hd, page_size);
  PA_REQUIRE(qkv && cos_table && sin_table && slots && kc && vc, "attn_decode_fused: a null operand");
  PA_REQUIRE(split_keys >= 32 && split_keys % 32 == 0, "attn_decode_fused: split of %d keys is not a multiple of 32", split_keys);
  PA_REQUIRE(max_splits >= 1 && max_splits <= 65535, "attn_decode_fused: %d splits", max_splits);
  PA_REQUIRE(max_splits == 1 || workspace, "attn_decode_fused: no workspace for %d splits", max_splits);
  float* part_o = workspace;
  float* part_ml = workspace ? workspace + (size_t)nseq * nh * max_splits * hd : nullptr;
  const FusedQkv fq{(const bf16*)qkv, q_weight, k_weight, cos_table, sin_table, slots, eps};
  const int shift = __builtin_ctz(page_size);
  if (hd == 64)
    return launch_decode<64, true>((hipStream_t)stream, nullptr, kc, vc, block_table, table_stride, seq_ids, cu_q,
                                   context_lens, out, part_o, part_ml, nseq, nh, nkv, shift, window, scale, softcap, nullptr,
                                   split_keys, max_splits, fq, ahead_list);
  return launch_decode<128, true>((hipStream_t)stream, nullptr, kc, vc, block_table, table_stride, seq_ids, cu_q,
                                  context_lens, out, part_o, part_ml, nseq, nh, nkv, shift, window, scale, softcap, nullptr,
                                  split_keys, max_splits, fq, ahead_list);
}

// min_prefix: the fewest keys any of the sequences has before its portion (0 if unknown): only a hint for how
// the work is cut.
// pa_attn_prefill with the cut given: paired (tiles in pairs), heads a wavefront (1, 2, 4), head groups a
// workgroup (1, 2), staged (keys through LDS); -1 leaves one to the launcher.  A cut the shape does not take is
// refused.  Every cut gives the same result up to rounding.
extern "C" int pa_attn_prefill_cut(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                                   int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                                   void* out, int nseq, int max_q_len, int min_prefix, int nh, int nkv, int hd,
                                   int page_size, int window, float scale, float softcap, int paired, int heads,
                                   int groups, int staged) {
  if (nseq == 0) return 0;
  if (int rc = check_common("attn_prefill", nseq, nh, nkv, page_size, table_stride, window)) return rc;
  PA_REQUIRE(max_q_len >= 1 && min_prefix >= 0, "attn_prefill: longest portion %d, shortest prefix %d", max_q_len, min_prefix);
  PA_REQUIRE(softcap >= 0.f, "attn_prefill: a score cap of %g is negative (0 means none)", (double)softcap);
  PrefillCut cut;
  cut.paired = paired, cut.heads = heads, cut.groups = groups, cut.staged = staged;
#define PA_CALL(HD)                                                                                                   \
  return launch_prefill<HD>((hipStream_t)stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, \
                            out, nseq, max_q_len, min_prefix, nh, nkv, __builtin_ctz(page_size), window, scale, softcap, nullptr, cut)
  PA_HD_SWITCH(hd, PA_CALL)
#undef PA_CALL
}

static int attn_prefill_entry(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                               int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                               void* out, int nseq, int max_q_len, int min_prefix, int nh, int nkv, int hd,
                               int page_size, int window, float scale, float softcap, const float* sink) {
  if (nseq == 0) return 0;
  if (int rc = check_common("attn_prefill", nseq, nh, nkv, page_size, table_stride, window)) return rc;
  PA_REQUIRE(max_q_len >= 1 && min_prefix >= 0, "attn_prefill: longest portion %d, shortest prefix %d", max_q_len, min_prefix);
  PA_REQUIRE(softcap >= 0.f, "attn_prefill: a score cap of %g is negative (0 means none)", (double)softcap);
#define PA_CALL(HD)                                                                                                   \
  return launch_prefill<HD>((hipStream_t)stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, \
                            out, nseq, max_q_len, min_prefix, nh, nkv, __builtin_ctz(page_size), window, scale, softcap, sink, \
                            PrefillCut{})
  PA_HD_SWITCH(hd, PA_CALL)
#undef PA_CALL
}

extern "C" int pa_attn_decode(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                              int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                              void* out, float* workspace, int nseq, int nh, int nkv, int hd, int page_size,
                              int window, float scale, float softcap, int split_keys, int max_splits) {
  return attn_decode_entry(stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out, workspace, nseq, nh,
                           nkv, hd, page_size, window, scale, softcap, nullptr, split_keys, max_splits);
}

extern "C" int pa_attn_prefill(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                               int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                               void* out, int nseq, int max_q_len, int min_prefix, int nh, int nkv, int hd,
                               int page_size, int window, float scale, float softcap) {
  return attn_prefill_entry(stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out, nseq, max_q_len,
                            min_prefix, nh, nkv, hd, page_size, window, scale, softcap, nullptr);
}

// The two with a sink per head (sink [nh], 32-bit, in the units of the scaled scores; null: none): a head's softmax
// divides by sum_j exp(s_j) + exp(sink_h).  The term joins a row's finished sums (in decode: after the splits are merged).
extern "C" int pa_attn_decode_sink(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                                   int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                                   void* out, float* workspace, int nseq, int nh, int nkv, int hd, int page_size,
                                   int window, float scale, float softcap, const float* sink, int split_keys,
                                   int max_splits) {
  return attn_decode_entry(stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out, workspace, nseq, nh,
                           nkv, hd, page_size, window, scale, softcap, sink, split_keys, max_splits);
}

extern "C" int pa_attn_prefill_sink(void* stream, const void* q, const void* kc, const void* vc, const int* block_table,
                                    int table_stride, const int* seq_ids, const int* cu_q, const int* context_lens,
                                    void* out, int nseq, int max_q_len, int min_prefix, int nh, int nkv, int hd,
                                    int page_size, int window, float scale, float softcap, const float* sink) {
  return attn_prefill_entry(stream, q, kc, vc, block_table, table_stride, seq_ids, cu_q, context_lens, out, nseq, max_q_len,
                            min_prefix, nh, nkv, hd, page_size, window, scale, softcap, sink);
}
