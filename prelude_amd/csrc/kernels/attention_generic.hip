// Paged causal attention for any mix of prompt portions and decode tokens,
// any head_dim up to 256, any page size, with or without a window, in 32-bit
// or bfloat16 storage.  All arithmetic is 32-bit on the vector ALU.  It is the
// attention of the true 32-bit path and the one that takes the sizes the MFMA
// kernels refuse.
//
// One workgroup of four wavefronts per (query token, query head), or per two
// query heads of a KV head (HEADS, below).  Keys are walked in chunks of 64
// anchored at absolute key positions that are multiples of 64, chunk c by
// wavefront c % 4, and the wavefronts' sums are merged in their order, so the
// order of every sum depends only on the query's position and window: the
// result for a token is bit-identical whether it arrives in a whole prompt, in
// a portion, or as a single decode token, and whatever pages hold its keys.
//
// What bounds it is the way from the caches to the registers: four lanes share
// a key (and, in the values, a dimension's sixteen keys), so that every load is
// 16 bytes a lane and 64 in a row.  With a key a lane and four bytes a load
// three decoding requests at a context of 150 took 64 us alone, 236 prompt
// tokens 141, 8 x 4,096 keys 1,660; with this and every load waited for before
// the next 30.9, 82 and 468; with two pieces ahead (FULL, below) 8.6, 46 and 118.
// A few requests take the time of one wavefront's instructions: without
// divisions by the page size and exchanges through LDS three at contexts of 26
// to 151 take 7.0 where they took 8.2.  Many tokens are bound by the number of
// loads (bfloat16 caches take as long as 32-bit ones): three prompts of 276
// tokens 53 us before, 37 with fewer registers and instructions, 30 with two
// heads a workgroup; one of 2,048 2,410, 2,329 and 1,241.
//
// K pages are [page, kv_head, offset, head_dim], V pages [page, kv_head, head_dim, offset].
//
// Formula: crates/prelude-core/src/models/qwen3.rs:276-370 and
// crates/prelude-core/src/ops/traits/attention.rs:10-99 (scores q.k * scale,
// key c visible to the query at position p when c <= p and, with a window of
// W keys, c > p - W; softmax in 32-bit; query head h reads KV head h / (nh/nkv)).  The reference's attention has
// no score cap (qwen3.rs:204); `softcap` > 0 bends the scaled scores to cap * tanh(s / cap) for mixers that want one.
#include "common.h"
#include "head_piece.h"
#include "api.h"

#include <type_traits>

namespace pa {

constexpr int kAttnWaves = 4;
constexpr int kAttnMaxHd = 256;
// Two heads of a KV head a workgroup from more (token, head) pairs than CUs on, up to head_dim 128 (above, two heads' registers
// leave a wavefront a SIMD).  16 heads of 128 in 32-bit, one head against two: a token each of 16 / 32 / 48 requests at a context of
// 150 7.4 against 8.3, 13.2 against 10.6 and 19.4 against 17.1 us, at 4,096 16 / 48 requests 120 against 130, 355 against 309;
// prompts of 16 / 64 / 512 / 2,048 tokens 5.0 against 5.9, 11.0 against 7.5, 174 against 109, 2,329 against 1,241.
constexpr long kOneHeadMostQueries = 256;

// Four elements in 32-bit: one load where `whole` (16 or 8 bytes, aligned), else the first `n` one by one and zeros.
template <typename T>
__device__ __forceinline__ f32x4 load_four(const T* at, bool whole, int n) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (whole) {
    if constexpr (sizeof(T) == 4) return *(const f32x4*)at;
    const bf16x4 x = *(const bf16x4*)at;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (float)x[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) v[e] = to_f32(at[e]);
  }
  return v;
}

template <typename T> struct FourOf { typedef f32x4 type; };
template <> struct FourOf<bf16> { typedef bf16x4 type; };
template <typename T> using Four = typename FourOf<T>::type;

// x / d for 0 <= x < 2^31 by a multiplication: with 2^(l-1) < d <= 2^l, x * (2^(31+l) / d + 1) / 2^(31+l), rounded down, is exact.
struct Divisor {
  unsigned times;
  int shift;
  __host__ explicit Divisor(int d) {
    int l = 0;
    while ((1LL << l) < d) ++l;
    shift = 31 + l;
    times = (unsigned)((1ULL << shift) / (unsigned)d + 1);
  }
  __device__ __forceinline__ int of(int x) const { return (int)(((unsigned long long)(unsigned)x * times) >> shift); }
};

constexpr int kRing = 2;   // pieces on their way; four are no faster, and at head_dim 256 slower (a wavefront a SIMD)

// What a step of single tokens brings in place of queries and written caches: the merged projection's rows, [nh + 2 nkv] heads a
// token, as they are (FUSED).  A token's key and value lie at `slots` (below 0: nowhere).
template <bool FUSED> struct RawRows {};
template <> struct RawRows<true> {
  const float *q_weight, *k_weight, *cos_table, *sin_table;
  const int* slots;
  float *k_cache, *v_cache;
  float eps;
};

// NI: head_dim in sixteens, rounded up; whole_k, whole_v: the rows of queries and keys, and of values, are aligned pieces of
// four.  FULL: both are, and head_dim is 16 NI.  A chunk is then eight pieces (four passes of keys, four groups of values),
// two always asked for ahead of their use, the first values before the softmax; left to itself the compiler waits for every
// load before it asks for the next (the same sums: with caches from memory, 16 heads of 128, three requests at a context of
// 150 30.9 -> 8.6 us, 236 prompt tokens 82 -> 46, 8 x 4,096 keys 468 -> 118, 2,048 tokens, which fill the chip, 2,537 -> 2,426).
//
// FUSED: every wavefront brings its query, and the key that the token adds, to unit RMS and turns them while its first pieces
// are on their way, a row half a wavefront (qknorm_rope_kv_wide_kernel's sums), and puts the new key and value where the caches would
// have them; the first head of a KV head writes them there, waited for by nobody.  What it saves is a launch; the rest of the path is
// that of the caches.  Inside a graph, us, in two launches / in one: 16 heads over 8 of 128, three contexts of 26 to 151 8.6 / 7.6,
// sixteen of 150 9.3 / 7.9, 32 over 8 at 1,003 keys 25.1 / 24.9, eight of 4,096 88.9 / 87.7; 14 over 2 of 64 10.4 / 9.4.  Four pieces
// on their way 7.8, 8.2, 25.8 and 94; a chunk's keys and dimensions over four wavefronts each (sixteen a workgroup, no fewer
// bytes through the compute unit) 8.8, 10.5, 26.6 and 101.
template <typename T, int NI, int HEADS, bool FUSED>
constexpr int kAttnOccupancy = FUSED ? 1 : HEADS == 1 ? (NI == 16 ? 2 : NI == 8 && sizeof(T) == 4 ? 3 : 4) : 2;

template <typename T, int NI, bool FULL, int HEADS, bool FUSED>
__global__ __launch_bounds__(kAttnWaves* kWave, (kAttnOccupancy<T, NI, HEADS, FUSED>)) void attn_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ seq_of_token,
    const int* __restrict__ positions, T* __restrict__ out, int nh, int nkv, int hd, int page_size, Divisor by_page, int window,
    float scale, float softcap, const float* __restrict__ sink, bool whole_k, bool whole_v, RawRows<FUSED> raw) {
  static_assert(!FUSED || (FULL && HEADS == 1 && sizeof(T) == 4 && NI <= 8), "a query and a key row a wavefront, 16 bytes a lane");
  if (FULL) {
    hd = NI * 16;
    whole_k = whole_v = true;
  }
  __shared__ float os[HEADS][kAttnWaves][NI * 16];
  __shared__ float ms[HEADS][kAttnWaves], ls[HEADS][kAttnWaves];
  __shared__ f32x4 ps[kAttnWaves][HEADS][kWave / 4];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int t = blockIdx.x, h = blockIdx.y * HEADS;
  const int hi = positions[t];
  const int lo = (window > 0 && hi - window + 1 > 0) ? hi - window + 1 : 0;
  const int kvh = h / (nh / nkv);
  const int* table = block_table + (size_t)seq_of_token[t] * table_stride;

  // queries and keys: lane (part, key) holds dimensions 16 i + 4 part + 0..3; values: lane (dim, part) dimension
  // 16 i + dim of keys 16 g + 4 part + 0..3 of the chunk
  const int part = lane / 16, key = lane % 16;
  const int vdim = lane / 4, vpart = lane % 4;
  f32x4 qv[HEADS][NI];
  constexpr int LPH = FUSED ? NI * 4 : kWave;                    // lanes a row
  __shared__ f32x4 rows[FUSED ? kAttnWaves : 1][3][LPH];         // the query, the new key and value, each wavefront's own
  const int sub = lane / LPH % 2, piece = lane % LPH;            // even ones take the query, odd ones the key
  f32x4 row, value, weight, cs, sn;
  int slot = -1;
  if constexpr (FUSED) {
    const T* token = q + (size_t)t * (nh + 2 * nkv) * hd + piece * 4;
    row = *(const f32x4*)(token + (sub ? nh + kvh : h) * hd);
    value = *(const f32x4*)(token + (nh + nkv + kvh) * hd);
    const float* w = sub ? raw.k_weight : raw.q_weight;
    weight = w ? *(const f32x4*)(w + piece * 4) : f32x4{1.f, 1.f, 1.f, 1.f};
    const size_t angle = (size_t)hi * (hd / 2) + piece % (LPH / 2) * 4;
    cs = *(const f32x4*)(raw.cos_table + angle), sn = *(const f32x4*)(raw.sin_table + angle);
    slot = raw.slots[t];
  } else {
    const T* qr = q + ((size_t)t * nh + h) * hd;
#pragma unroll
    for (int a = 0; a < HEADS; ++a)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int d = i * 16 + part * 4;
        qv[a][i] = d < hd ? load_four(qr + a * hd + d, whole_k, hd - d) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }

  const auto pages_of = [&](int c) { return by_page.of(c); };
  float m[HEADS], l[HEADS] = {}, o[HEADS][NI] = {};
#pragma unroll
  for (int a = 0; a < HEADS; ++a) m[a] = -INFINITY;
  const int begin = (lo / kWave + ((wave - lo / kWave) & (kAttnWaves - 1))) * kWave;
  for (int c0 = begin; c0 <= hi; c0 += kAttnWaves * kWave) {
    float s[HEADS] = {};
    Four<T> ring[kRing][NI];
    int kpage[4], vpage[4];
    // piece n of a chunk: four passes of sixteen keys, then four groups of values
    auto fetch = [&](int n) {
      if (n < 4) {
        const int c = min(max(c0 + n * 16 + key, lo), hi);      // keys that are not seen: any that is
        const T* kr = k_cache + (((size_t)kpage[n] * nkv + kvh) * page_size + (c - pages_of(c) * page_size)) * hd + part * 4;
#pragma unroll
        for (int i = 0; i < NI; ++i) ring[n % kRing][i] = *(const Four<T>*)(kr + i * 16);
      } else {                                                  // four keys lie in one page; beyond what is seen: the page of one that is
        const int c = c0 + (n - 4) * 16 + vpart * 4;
        const T* vr = v_cache + (((size_t)vpage[n - 4] * nkv + kvh) * hd + vdim) * page_size + (c - pages_of(c) * page_size);
#pragma unroll
        for (int i = 0; i < NI; ++i) ring[n % kRing][i] = *(const Four<T>*)(vr + (size_t)i * 16 * page_size);
      }
      __builtin_amdgcn_sched_barrier(0);                        // asked for here, whatever registers it holds
    };
    if constexpr (FULL) {
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        kpage[n] = table[pages_of(min(max(c0 + n * 16 + key, lo), hi))];
        vpage[n] = table[pages_of(min(max(c0 + n * 16 + vpart * 4, lo), hi))];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < kRing; ++n) fetch(n);
    }
    if constexpr (FUSED) {
      if (c0 == begin) {
        float x[4], w[4], c[4], s_[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = row[e], w[e] = weight[e], c[e] = cs[e], s_[e] = sn[e];
        norm_turn_piece<LPH>(x, w, c, s_, (sub ? raw.k_weight : raw.q_weight) != nullptr, raw.eps, piece);
        rows[wave][sub][piece] = f32x4{x[0], x[1], x[2], x[3]};
        rows[wave][2][piece] = value;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < NI; ++i) qv[0][i] = rows[wave][0][i * 4 + part];
      }
    }
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
      f32x4 dot[HEADS] = {};
      if constexpr (FULL) {
        if constexpr (FUSED) {
          const int k0 = c0 + pass * 16;
          if (hi >= k0 && hi < k0 + 16 && k0 + key == hi && kpage[pass] * page_size + hi - pages_of(hi) * page_size == slot) {
#pragma unroll
            for (int i = 0; i < NI; ++i) ring[pass % kRing][i] = rows[wave][1][i * 4 + part];
          }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int a = 0; a < HEADS; ++a) dot[a][e] = fmaf(qv[a][i][e], (float)ring[pass % kRing][i][e], dot[a][e]);
        fetch(pass + kRing);
      } else {
        const int c = min(max(c0 + pass * 16 + key, lo), hi);     // keys that are not seen: any that is
        const int page = table[pages_of(c)];
        const T* kr = k_cache + (((size_t)page * nkv + kvh) * page_size + (c - pages_of(c) * page_size)) * hd;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int d = i * 16 + part * 4;
          if (d < hd) {
            const f32x4 kv = load_four(kr + d, whole_k, hd - d);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int a = 0; a < HEADS; ++a) dot[a][e] = fmaf(qv[a][i][e], kv[e], dot[a][e]);
          }
        }
      }
#pragma unroll
      for (int a = 0; a < HEADS; ++a) {
        float sum = (dot[a][0] + dot[a][1]) + (dot[a][2] + dot[a][3]);
        unsigned u = __float_as_uint(sum);                       // from the lanes 16 and 32 away
        const auto near = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        u = __float_as_uint(__uint_as_float(near[0]) + __uint_as_float(near[1]));
        const auto far = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        sum = __uint_as_float(far[0]) + __uint_as_float(far[1]);
        if (part == pass) s[a] = sum;                            // lane by lane: its own key of the 64
      }
    }
    const int c = c0 + lane;
    const bool valid = c >= lo && c <= hi;
#pragma unroll
    for (int a = 0; a < HEADS; ++a) {
      s[a] *= scale;
      if (softcap != 0.f) s[a] = softcap * tanhf(s[a] / softcap);   // scores bent into (-cap, cap)
      if (!valid) s[a] = -INFINITY;
      const float m_new = fmaxf(m[a], wave_max(s[a]));
      const float from = m_new == -INFINITY ? 0.f : m_new;  // no finite score in this wavefront's keys yet: every p is 0
      const float p = valid ? expf(s[a] - from) : 0.f;
      const float alpha = expf(m[a] - from);   // exp(-inf) = 0 on the first chunk
      l[a] = l[a] * alpha + wave_sum(p);
#pragma unroll
      for (int i = 0; i < NI; ++i) o[a][i] *= alpha;
      reinterpret_cast<float*>(ps[wave][a])[lane] = p;
      m[a] = m_new;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int j = g * 16 + vpart * 4;                         // the lane's four keys
      f32x4 pj[HEADS];
#pragma unroll
      for (int a = 0; a < HEADS; ++a) pj[a] = ps[wave][a][j / 4];
      if constexpr (FULL) {
        if constexpr (FUSED) {
          const int k0 = c0 + g * 16, at = hi - c0 - j;
          if (hi >= k0 && hi < k0 + 16 && at >= 0 && at < 4 && vpage[g] * page_size + hi - pages_of(hi) * page_size == slot) {
            const float* fresh = reinterpret_cast<const float*>(rows[wave][2]);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) ring[g % kRing][i][e] = e == at ? fresh[i * 16 + vdim] : ring[g % kRing][i][e];
          }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {                         // what lies beside the keys may be anything
            const float v = c0 + j + e >= lo && c0 + j + e <= hi ? (float)ring[g % kRing][i][e] : 0.f;
#pragma unroll
            for (int a = 0; a < HEADS; ++a) o[a][i] = fmaf(pj[a][e], v, o[a][i]);
          }
        if (g + kRing < 4) fetch(g + 4 + kRing);
        continue;
      }
      if (c0 + j > hi || c0 + j + 3 < lo) continue;
      if (whole_v) {                                            // four keys lie in one page; beyond what is seen: the page of one that is
        const int page = table[pages_of(min(max(c0 + j, lo), hi))];
        const T* vr = v_cache + ((size_t)page * nkv + kvh) * hd * page_size + (c0 + j - pages_of(c0 + j) * page_size);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int d = i * 16 + vdim;
          if (d >= hd) continue;
          const f32x4 vv = load_four(vr + (size_t)d * page_size, true, 4);
#pragma unroll
          for (int e = 0; e < 4; ++e)                           // what lies beside the keys may be anything
#pragma unroll
            for (int a = 0; a < HEADS; ++a) o[a][i] = fmaf(pj[a][e], c0 + j + e >= lo && c0 + j + e <= hi ? vv[e] : 0.f, o[a][i]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int cj = min(max(c0 + j + e, lo), hi);
          const T* vr = v_cache + ((size_t)table[pages_of(cj)] * nkv + kvh) * hd * page_size + (cj - pages_of(cj) * page_size);
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const int d = i * 16 + vdim;
            if (d >= hd) continue;
            const float v = cj == c0 + j + e ? to_f32(vr[(size_t)d * page_size]) : 0.f;
#pragma unroll
            for (int a = 0; a < HEADS; ++a) o[a][i] = fmaf(pj[a][e], v, o[a][i]);
          }
        }
      }
    }
    __builtin_amdgcn_wave_barrier();                            // the next chunk's weights go where these were read
    if constexpr (FUSED) {
      if (slot >= 0 && hi < c0 + kWave && h % (nh / nkv) == 0) {
        const int page = pages_of(slot), off = slot - page * page_size;
        const size_t head = ((size_t)page * nkv + kvh) * page_size * hd;
        if (lane < LPH) *(f32x4*)(raw.k_cache + head + (size_t)off * hd + lane * 4) = rows[wave][1][lane];
#pragma unroll
        for (int d = lane; d < NI * 16; d += kWave)
          raw.v_cache[head + (size_t)d * page_size + off] = reinterpret_cast<const float*>(rows[wave][2])[d];
      }
    }
  }
#pragma unroll
  for (int a = 0; a < HEADS; ++a) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float v = o[a][i];
      v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));   // one lane away
      v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, true));   // two
      if (vpart == 0) os[a][wave][i * 16 + vdim] = v;
    }
    if (lane == 0) {
      ms[a][wave] = m[a];
      ls[a][wave] = l[a];
    }
  }
  __syncthreads();
  for (int at = threadIdx.x; at < HEADS * hd; at += kAttnWaves * kWave) {
    const int a = HEADS > 1 && at >= hd ? 1 : 0, d = at - a * hd;
    const float most = fmaxf(fmaxf(ms[a][0], ms[a][1]), fmaxf(ms[a][2], ms[a][3]));
    float total = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      if (ls[a][w] == 0.f && ms[a][w] == -INFINITY) continue;   // a wavefront without a chunk
      const float alpha = expf(ms[a][w] - most);
      total = fmaf(ls[a][w], alpha, total);
      sum = fmaf(os[a][w][d], alpha, sum);
    }
    float inv = 1.0f / total;
    if (sink) {   // one more term exp(sink) of the denominator that brings no value
      const float m_fin = fmaxf(most, sink[h + a]);
      const float alpha = expf(most - m_fin);
      inv = alpha / (total * alpha + expf(sink[h + a] - m_fin));
    }
    out[((size_t)t * nh + h + a) * hd + d] = from_f32<T>(sum * inv);
  }
}

}  // namespace pa

using namespace pa;

static int attn_generic_launch(void* stream, int dtype, const void* q, const void* k_cache, const void* v_cache,
                               const int* block_table, int table_stride, const int* seq_of_token,
                               const int* positions, void* out, int tokens, int nh, int nkv, int hd, int page_size,
                               int window, float scale, float softcap, const float* sink) {
  if (tokens == 0) return 0;
  PA_REQUIRE(tokens > 0 && nh > 0 && nkv > 0 && page_size > 0 && table_stride > 0,
             "attn_generic: bad sizes tokens=%d nh=%d nkv=%d page=%d table_stride=%d", tokens, nh, nkv, page_size,
             table_stride);
  PA_REQUIRE(nh % nkv == 0, "attn_generic: %d query heads are not a multiple of %d KV heads", nh, nkv);
  PA_REQUIRE(hd > 0 && hd <= kAttnMaxHd, "attn_generic: head_dim %d is outside 1..%d", hd, kAttnMaxHd);
  PA_REQUIRE(window >= 0, "attn_generic: window %d is negative (0 means none)", window);
  PA_REQUIRE(softcap >= 0.f, "attn_generic: a score cap of %g is negative (0 means none)", (double)softcap);
  const size_t piece = dtype == kF32 ? 16 : 8;   // four elements
  const bool whole_k = hd % 4 == 0 && ((uintptr_t)q | (uintptr_t)k_cache) % piece == 0;
  const bool whole_v = page_size % 4 == 0 && (uintptr_t)v_cache % piece == 0;
  hipStream_t st = (hipStream_t)stream;
  const Divisor by_page(page_size);
  const bool pairs = nh / nkv % 2 == 0 && (long)tokens * nh > kOneHeadMostQueries;
  auto launch = [&](auto zero, auto ni, auto full) {
    typedef decltype(zero) T;
    constexpr int NI = decltype(ni)::value;
    constexpr bool FULL = decltype(full)::value;
    const auto run = [&](auto* kernel, dim3 grid) {
      hipLaunchKernelGGL(kernel, grid, dim3(kAttnWaves * kWave), 0, st, (const T*)q, (const T*)k_cache, (const T*)v_cache, block_table,
                         table_stride, seq_of_token, positions, (T*)out, nh, nkv, hd, page_size, by_page, window, scale, softcap, sink,
                         whole_k, whole_v, RawRows<false>{});
    };
    if constexpr (NI <= 8)
      if (pairs) return run(&attn_generic_kernel<T, NI, FULL, 2, false>, dim3(tokens, nh / 2));
    run(&attn_generic_kernel<T, NI, FULL, 1, false>, dim3(tokens, nh));
  };
  auto by_fit = [&](auto zero, auto ni) {
    if (whole_k && whole_v && hd == 16 * decltype(ni)::value) launch(zero, ni, std::true_type());
    else launch(zero, ni, std::false_type());
  };
  auto by_width = [&](auto zero) {
    if (hd <= 64) by_fit(zero, std::integral_constant<int, 4>());
    else if (hd <= 128) by_fit(zero, std::integral_constant<int, 8>());
    else by_fit(zero, std::integral_constant<int, 16>());
  };
  if (dtype == kF32) by_width(0.f);
  else if (dtype == kBF16) by_width(bf16(0.f));
  else return pa::fail("attn_generic: unknown element type code %d", dtype);
  return check_launch("attn_generic");
}

extern "C" int pa_attn_generic(void* stream, int dtype, const void* q, const void* k_cache, const void* v_cache,
                               const int* block_table, int table_stride, const int* seq_of_token,
                               const int* positions, void* out, int tokens, int nh, int nkv, int hd, int page_size,
                               int window, float scale, float softcap) {
  return attn_generic_launch(stream, dtype, q, k_cache, v_cache, block_table, table_stride, seq_of_token, positions, out, tokens,
                             nh, nkv, hd, page_size, window, scale, softcap, nullptr);
}

// The same with a sink per head (sink [nh], 32-bit, in the units of the scaled scores): the softmax divides by
// sum_j exp(s_j) + exp(sink_h); nothing is attended to through it.
extern "C" int pa_attn_generic_sink(void* stream, int dtype, const void* q, const void* k_cache, const void* v_cache,
                                    const int* block_table, int table_stride, const int* seq_of_token,
                                    const int* positions, void* out, int tokens, int nh, int nkv, int hd, int page_size,
                                    int window, float scale, float softcap, const float* sink) {
  return attn_generic_launch(stream, dtype, q, k_cache, v_cache, block_table, table_stride, seq_of_token, positions, out, tokens,
                             nh, nkv, hd, page_size, window, scale, softcap, sink);
}

// Whether pa_attn_generic_fused takes a step of `tokens` single tokens: heads of 64 or 128 turned over their whole width, pages of whole
// fours, and no more (token, head) pairs than one head a workgroup takes.
extern "C" int pa_attn_generic_fused_supports(int tokens, int nh, int nkv, int hd, int rot, int page_size) {
  return tokens > 0 && nkv > 0 && nh > 0 && nh % nkv == 0 && (hd == 64 || hd == 128) && rot == hd && page_size > 0 && page_size % 4 == 0 &&
         (long)tokens * nh <= kOneHeadMostQueries;
}

// pa_qknorm_rope_kv and pa_attn_generic of a 32-bit step in which every sequence feeds one token, in one launch and to the bit: qkv
// [tokens, nh + 2 nkv, hd] the merged projection, whose keys and values go to `slots` of the caches and are attended to.
extern "C" int pa_attn_generic_fused(void* stream, const float* qkv, const float* q_weight, const float* k_weight, const float* cos_table,
                                     const float* sin_table, const int* slots, float eps, float* k_cache, float* v_cache,
                                     const int* block_table, int table_stride, const int* seq_of_token, const int* positions, float* out,
                                     int tokens, int nh, int nkv, int hd, int page_size, int window, float scale, float softcap) {
  if (tokens == 0) return 0;
  PA_REQUIRE(pa_attn_generic_fused_supports(tokens, nh, nkv, hd, hd, page_size) && table_stride > 0,
             "attn_generic_fused: sizes tokens=%d nh=%d nkv=%d hd=%d page=%d table_stride=%d are not taken", tokens, nh, nkv, hd, page_size,
             table_stride);
  PA_REQUIRE(qkv && cos_table && sin_table && slots && k_cache && v_cache && block_table && seq_of_token && positions && out,
             "attn_generic_fused: an operand is missing");
  PA_REQUIRE((((uintptr_t)qkv | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)cos_table | (uintptr_t)sin_table | (uintptr_t)k_cache |
               (uintptr_t)v_cache) & 15) == 0, "attn_generic_fused: operands are not 16-byte aligned");
  PA_REQUIRE(window >= 0, "attn_generic_fused: window %d is negative (0 means none)", window);
  PA_REQUIRE(softcap >= 0.f, "attn_generic_fused: a score cap of %g is negative (0 means none)", (double)softcap);
  const RawRows<true> raw{q_weight, k_weight, cos_table, sin_table, slots, k_cache, v_cache, eps};
  const auto launch = [&](auto* kernel) {
    hipLaunchKernelGGL(kernel, dim3(tokens, nh), dim3(kAttnWaves * kWave), 0, (hipStream_t)stream, qkv, (const float*)k_cache,
                       (const float*)v_cache, block_table, table_stride, seq_of_token, positions, out, nh, nkv, hd, page_size,
                       Divisor(page_size), window, scale, softcap, (const float*)nullptr, true, true, raw);
  };
  if (hd == 64) launch(&attn_generic_kernel<float, 4, true, 1, true>);
  else launch(&attn_generic_kernel<float, 8, true, 1, true>);
  return check_launch("attn_generic_fused");
}
