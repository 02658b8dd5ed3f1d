// Recurrent mixers whose state is a matrix per (request, head) that decays by one number a token:
//
//   S_t = a_t S_(t-1) + b_t k_t v_t^T          S [dim, vdim], 32-bit, one per (request, head), kept in a state slot
//   n_t = a_t n_(t-1) + b_t k_t                n [dim], where the design keeps one
//   o_t = S_t^T q_t + skip_h v_t,   den_t = n_t . q_t        (q times a constant on its way in), 32-bit
//
// with a_t = exp(la_t) and b_t one number per token and head, made in 32-bit from the projections by
//   ssd gates     b = softplus(z + bias), la = -exp(a_log) b                                            (Mamba-2)
//   mlstm gates   i = c tanh((z_i + bias_i) / c), f = log sigmoid(c tanh((z_f + bias_f) / c)), and a running maximum m (zero
//                 at a request's start): m_t = max(f + m_(t-1), i), la = f + m_(t-1) - m_t, b = exp(i - m_t); the reader of
//                 den also gets exp(-m_t)                                                                (xLSTM's mLSTM)
//
// q, k [tokens, heads / group, dim] (head h reads q/k head h / group) and v [tokens, heads, vdim] lie inside one row per
// token (stride ld).  A request's portions may be cut anywhere; the state carries over.
//
//   pa_decay_scan          the recurrence as it stands, token by token, on the vector ALU, for any sizes and both types
//   pa_decay_scan_step     single tokens, gates included
//   pa_decay_scan_chunked  portions, bfloat16, on the matrix cores, in chunks of 64 tokens.  With c_i the sum of la up to
//                          token i of a chunk and S_b the state in front of it,
//
//                            o_i  = sum_{j <= i} e^(c_i - c_j) b_j (q_i . k_j) v_j  +  e^(c_i) S_b^T q_i
//                            S_b' = e^(c_n) S_b + U,    U = sum_j e^(c_n - c_j) b_j k_j v_j^T
//
//                          A workgroup walks a segment of up to four chunks with the state in registers.  Sequences of more than one: (1) every
//                          segment makes its U, (2) one pass over the segments of a sequence turns the U into the states in front of them, (3)
//                          every segment makes its outputs, and the last the slot's state.  Segments begin with the portion, so a sequence's
//                          numbers do not depend on what else is in the step.  The sums c are 64-bit, so a difference of two of them is
//                          exact to 32-bit whatever came before.  What is not a stored bfloat16 number already -- the weights of the first
//                          sum, the scaled keys of U, the state -- takes part as the sum of two bfloat16 numbers (a product with 16 bits of
//                          mantissa, added up in 32-bit).
#include "common.h"
#include "api.h"
#include "attention_mfma_core.h"

namespace pa {

constexpr int kScanCols = 64;      // value columns a workgroup of the token-by-token kernels
constexpr int kScanTokens = 16;    // tokens staged at a time
constexpr int kScanThreads = 256;
constexpr int kScanChunk = 64;
constexpr int kScanMostChunks = 4;  // chunks a workgroup of the chunked kernels walks at most

template <typename T>
struct ScanArgs {
  const T* p;
  size_t ld;
  int q_off, k_off, v_off;
  int heads, group, dim, vdim;
  const float* la;     // [tokens, heads]
  const float* b;      // [tokens, heads]
  float* s;            // [slots, heads, dim, vdim]
  float* n;            // [slots, heads, dim], or null
  const float* skip;   // [heads], or null
  float q_scale;
  const int* slots;
  const int* cu_q;
  float* out;          // [tokens, heads, vdim]
  float* den;          // [tokens, heads], or null
};

__device__ __forceinline__ float scan_softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float scan_log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float scan_capped(float z, float cap) { return cap * tanhf(z / cap); }

// ---- gates of portions -------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void ssd_gates_kernel(const T* __restrict__ p, size_t ld, int off, const float* __restrict__ bias,
                                                        const float* __restrict__ a_log, float* __restrict__ la,
                                                        float* __restrict__ b, size_t total, int heads) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / heads;
  const int h = (int)(i % heads);
  const float dt = scan_softplus(to_f32(p[t * ld + off + h]) + bias[h]);
  b[i] = dt;
  la[i] = -expf(a_log[h]) * dt;
}

// A workgroup a (head, sequence of at least min_len tokens), 1,024 tokens at a time, a thread a token.  A token is the map
// m -> max(f + m, i), and maps compose: (f1, i1) and then (f2, i2) is (f1 + f2, max(i1 + f2, i2)).
constexpr int kGateThreads = 1024;

template <typename T>
__global__ __launch_bounds__(kGateThreads) void mlstm_gates_kernel(const T* __restrict__ p, size_t ld, int i_off, int f_off,
                                                                   const float* __restrict__ i_bias, const float* __restrict__ f_bias,
                                                                   float cap, float* __restrict__ m_state, int copies,
                                                                   const int* __restrict__ state_slots, const int* __restrict__ cu_q,
                                                                   float* __restrict__ la, float* __restrict__ b,
                                                                   float* __restrict__ floor_out, int heads, int min_len) {
  constexpr int kWaves = kGateThreads / kWave;
  __shared__ float wave_f[2][kWaves], wave_i[2][kWaves];
  const int h = blockIdx.x, seq = blockIdx.y, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int row0 = cu_q[seq], row1 = cu_q[seq + 1];
  const int slot = state_slots[seq];
  if (slot < 0 || row1 - row0 < min_len || row1 <= row0) return;   // the same for the whole workgroup
  float* ms = m_state + ((size_t)slot * heads + h) * copies;
  float m = ms[0];
  const float ib = i_bias[h], fb = f_bias[h];
  int buf = 0;
  for (int t0 = row0; t0 < row1; t0 += kGateThreads, buf ^= 1) {
    const int t = t0 + threadIdx.x;
    const bool live = t < row1;
    const T* z = p + (size_t)(live ? t : row1 - 1) * ld + h;
    const float zi = to_f32(z[i_off]), zf = to_f32(z[f_off]);
    const float ig = live ? scan_capped(zi + ib, cap) : -INFINITY;
    const float fg = live ? scan_log_sigmoid(scan_capped(zf + fb, cap)) : 0.f;
    float A = fg, B = ig;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const float Ao = __shfl_up(A, o, kWave), Bo = __shfl_up(B, o, kWave);
      if (lane >= o) {
        B = fmaxf(Bo + A, B);
        A += Ao;
      }
    }
    if (lane == kWave - 1) {
      wave_f[buf][wave] = A;
      wave_i[buf][wave] = B;
    }
    __syncthreads();               // (two buffers: the next block's sums do not meet this one's readers)
    float mine = m;                // the maximum in front of this wavefront's tokens, and behind the block's
    for (int w = 0; w < kWaves; ++w) {
      if (w == wave) mine = m;
      m = fmaxf(wave_f[buf][w] + m, wave_i[buf][w]);
    }
    const float mt = fmaxf(A + mine, B);
    float before = __shfl_up(mt, 1, kWave);
    if (lane == 0) before = mine;
    if (live) {
      const size_t at = (size_t)t * heads + h;
      la[at] = fg + before - mt;
      b[at] = expf(ig - mt);
      floor_out[at] = expf(-mt);
    }
  }
  __syncthreads();                 // every thread has read the slot
  for (int i = threadIdx.x; i < copies; i += kGateThreads) ms[i] = m;
}

// ---- token by token ----------------------------------------------------------------------------------------------------
// Grid (tiles of 64 value columns, and one more for n where there is one; heads; sequences of at least min_len tokens).  A lane
// keeps a quarter of the rows of S (R of them) for one column in registers: the 16-lane rows of a wavefront are the
// quarters, whose dot products are added across them.
template <typename T, int R>
__global__ __launch_bounds__(kScanThreads) void decay_scan_kernel(ScanArgs<T> a, int min_len) {
  constexpr int kQuarter = R + 4;
  __shared__ __align__(16) float qs[kScanTokens][4 * kQuarter];
  __shared__ __align__(16) float ks[kScanTokens][4 * kQuarter];
  __shared__ float vs[kScanTokens][kScanCols];
  __shared__ float as[kScanTokens], bs[kScanTokens];
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int dp = lane / 16, cl = 16 * w + lane % 16;
  const int h = blockIdx.y, seq = blockIdx.z;
  const int row0 = a.cu_q[seq], row1 = a.cu_q[seq + 1];
  const int slot = a.slots[seq];
  if (slot < 0 || row1 - row0 < min_len || row1 <= row0) return;   // the same for the whole workgroup
  const int vt = (a.vdim + kScanCols - 1) / kScanCols;
  const bool is_n = (int)blockIdx.x == vt;
  const int c0 = is_n ? 0 : blockIdx.x * kScanCols;
  const int width = is_n ? 1 : a.vdim;
  const int col = c0 + cl;
  const bool live = col < width;
  float* sp = is_n ? a.n + ((size_t)slot * a.heads + h) * a.dim : a.s + ((size_t)slot * a.heads + h) * a.dim * a.vdim;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = dp * R + r;
    S[r] = (live && d < a.dim) ? sp[(size_t)d * width + col] : 0.f;
  }
  const T* qp = a.p + a.q_off + (size_t)(h / a.group) * a.dim;
  const T* kp = a.p + a.k_off + (size_t)(h / a.group) * a.dim;
  const T* vp = a.p + a.v_off + (size_t)h * a.vdim;
  const float skip = (a.skip && !is_n) ? a.skip[h] : 0.f;
  for (int t0 = row0; t0 < row1; t0 += kScanTokens) {
    const int n = row1 - t0 < kScanTokens ? row1 - t0 : kScanTokens;
    __syncthreads();
    for (int e = threadIdx.x; e < kScanTokens * 4 * R; e += kScanThreads) {
      const int t = e / (4 * R), d = e % (4 * R);
      const bool on = t < n && d < a.dim;
      const size_t at = (size_t)(t0 + t) * a.ld + d;
      const int to = (d / R) * kQuarter + d % R;
      qs[t][to] = on ? to_f32(qp[at]) * a.q_scale : 0.f;
      ks[t][to] = on ? to_f32(kp[at]) : 0.f;
    }
    for (int e = threadIdx.x; e < kScanTokens * kScanCols; e += kScanThreads) {
      const int t = e / kScanCols, c = e % kScanCols;
      const bool on = t < n && c0 + c < width;
      vs[t][c] = on ? (is_n ? 1.f : to_f32(vp[(size_t)(t0 + t) * a.ld + c0 + c])) : 0.f;
    }
    if ((int)threadIdx.x < n) {
      const size_t at = (size_t)(t0 + threadIdx.x) * a.heads + h;
      as[threadIdx.x] = expf(a.la[at]);
      bs[threadIdx.x] = a.b[at];
    }
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      const float al = as[t], v = vs[t][cl], bv = bs[t] * v;
      float acc = 0.f;
#pragma unroll
      for (int r = 0; r < R; r += 4) {
        const f32x4 q4 = *reinterpret_cast<const f32x4*>(&qs[t][dp * kQuarter + r]);
        const f32x4 k4 = *reinterpret_cast<const f32x4*>(&ks[t][dp * kQuarter + r]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[r + e] = fmaf(al, S[r + e], k4[e] * bv);
          acc = fmaf(S[r + e], q4[e], acc);
        }
      }
      const float sum = xor_sum16_32(acc);
      if (dp == 0 && live) {
        const size_t at = (size_t)(t0 + t) * a.heads + h;
        if (is_n) a.den[at] = sum;
        else a.out[at * a.vdim + col] = fmaf(skip, v, sum);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = dp * R + r;
    if (live && d < a.dim) sp[(size_t)d * width + col] = S[r];
  }
}

// How a single token's gates are made on the way in.
template <typename T>
struct StepGates {
  const T* z;               // rows of stride z_ld that hold the heads' gate inputs
  size_t z_ld;
  int z_off, f_off;         // their columns (mlstm: of i and f)
  const float* bias;        // [heads] (mlstm: of i)
  const float* f_bias;      // mlstm
  const float* a_log;       // ssd
  float cap;                // mlstm
  float* m;                 // mlstm: [slots, heads, copies], a copy of the running maximum per column tile
  int copies;
  float* floor_out;         // mlstm: exp(-m) [tokens, heads]
};

// Sequences of exactly one token.  Grid as above; a wavefront owns a quarter of the rows, a lane a column: a row's 64 columns
// are one run of memory, and all of a lane's rows are asked for at once.
// WHOLE: dim is 4 R, so that every row of a wavefront's quarter exists and its addresses are the wavefront's.  A few sequences are
// bound by a wavefront's path: with the gates computed while the state is on its way, and no address or condition a lane and row, three
// sequences of 64 heads of 128 x 64 take 5.2 us where they took 7.5 (one 4.6 and 6.6, sixteen 17.7 and 19.0, 134 MB), of 8 mLSTM heads of
// 128 x 256 5.2 (7.1).
template <typename T, int R, bool MLSTM, bool WHOLE>
__global__ __launch_bounds__(kScanThreads) void decay_scan_step_kernel(ScanArgs<T> a, StepGates<T> g) {
  __shared__ float qs[4 * R], ks[4 * R];
  __shared__ float part[4][kScanCols];
  const int w = WHOLE ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) : threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int h = blockIdx.y, seq = blockIdx.z;
  const int row = a.cu_q[seq];
  const int slot = a.slots[seq];
  if (slot < 0 || a.cu_q[seq + 1] - row != 1) return;   // the same for the whole workgroup
  const int vt = (a.vdim + kScanCols - 1) / kScanCols;
  const bool is_n = (int)blockIdx.x == vt;
  const int col = (is_n ? 0 : blockIdx.x * kScanCols) + lane;
  const int width = is_n ? 1 : a.vdim;
  const bool live = col < width;
  float* sp = is_n ? a.n + ((size_t)slot * a.heads + h) * a.dim : a.s + ((size_t)slot * a.heads + h) * a.dim * a.vdim;
  const unsigned at_col = live ? col : width - 1;               // (a row's address is the wavefront's, the column the lane's)
  // what the gates and the products need first, then the state: loads come back in the order in which they were asked for
  const T* src = a.p + (size_t)row * a.ld;
  const int qd = (int)threadIdx.x < a.dim ? threadIdx.x : a.dim - 1;
  const T q = src[a.q_off + (size_t)(h / a.group) * a.dim + qd], k = src[a.k_off + (size_t)(h / a.group) * a.dim + qd];
  const T value = src[a.v_off + (size_t)h * a.vdim + (live && !is_n ? col : a.vdim - 1)];
  const T* zr = g.z + (size_t)row * g.z_ld + h;
  const T z = zr[g.z_off], zf = zr[MLSTM ? g.f_off : g.z_off];
  const float bias = g.bias[h], last = MLSTM ? g.f_bias[h] : g.a_log[h];
  float* mp = MLSTM ? g.m + ((size_t)slot * a.heads + h) * g.copies + blockIdx.x : nullptr;
  const float m = MLSTM ? *mp : 0.f;
  __builtin_amdgcn_sched_barrier(0);
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = w * R + r;
    s[r] = (sp + (size_t)(WHOLE || d < a.dim ? d : a.dim - 1) * width)[at_col];
  }
  __builtin_amdgcn_sched_barrier(0);
  if ((int)threadIdx.x < 4 * R) {
    qs[threadIdx.x] = to_f32(q) * a.q_scale;
    ks[threadIdx.x] = to_f32(k);
  }
  const float v = is_n ? 1.f : to_f32(value);
  float al, b, m_new = 0.f;
  if (MLSTM) {
    const float ig = scan_capped(to_f32(z) + bias, g.cap);
    const float fg = scan_log_sigmoid(scan_capped(to_f32(zf) + last, g.cap));
    m_new = fmaxf(fg + m, ig);
    al = expf(fg + m - m_new);
    b = expf(ig - m_new);
  } else {
    b = scan_softplus(to_f32(z) + bias);
    al = expf(-expf(last) * b);
  }
  asm volatile("" ::"v"(al), "v"(b));   // the gates on this side of the barrier: under the state's way, and the running maximum read
  __syncthreads();
  if (MLSTM && threadIdx.x == 0) {   // behind the barrier: every thread has read its copy
    *mp = m_new;
    if (is_n) g.floor_out[(size_t)row * a.heads + h] = expf(-m_new);
  }
  const float bv = b * v;
  float acc = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int d = w * R + r;
    s[r] = fmaf(al, s[r], ks[d] * bv);
    if (WHOLE || d < a.dim) acc = fmaf(s[r], qs[d], acc);
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int d = w * R + r;
      if (WHOLE || d < a.dim) (sp + (size_t)d * width)[at_col] = s[r];
    }
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0 && live) {
    const float sum = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    const size_t at = (size_t)row * a.heads + h;
    if (is_n) a.den[at] = sum;
    else a.out[at * a.vdim + col] = fmaf(a.skip ? a.skip[h] : 0.f, v, sum);
  }
}

// ---- portions in chunks, on the matrix cores ---------------------------------------------------------------------------
// How a sequence of `chunks` chunks is cut into segments, a workgroup for each of them and 64 columns of a head's state (`parts` for all heads): of one chunk
// where that leaves few workgroups, of four where there are many.  By the sequence alone, so that its numbers do not depend on what else is in the step.
struct ScanSegments {
  int chunks, each, count;
  __host__ __device__ __forceinline__ ScanSegments(int len, int parts) {
    chunks = (len + kScanChunk - 1) / kScanChunk;
    each = chunks <= kScanMostChunks ? kScanMostChunks : (int)(((long)chunks * parts + 85) / 170);
    each = each < 1 ? 1 : (each > kScanMostChunks ? kScanMostChunks : each);
    count = (chunks + each - 1) / each;
  }
};
// Where segment j of the z-th listed sequence, which starts at packed row row0, keeps its state: every sequence adds at most one
// partial chunk, so the index is different for every segment of the launch and below tokens / 64 + sequences.
__device__ __forceinline__ size_t scan_segment_index(int row0, int z, int j) { return (size_t)(row0 / kScanChunk + z + j); }

// LDS of the kernel below: rows of 64 tokens, 128 bytes each, in eight pieces of eight tokens whose places are turned by the row, so that
// operands (sixteen rows' pieces of the same tokens) and, of those that are written by pairs of tokens, eight columns lie in different banks as far
// as that leaves the rows of a thread's eight columns at fixed distances.
// The weights, [query][key].
__device__ __forceinline__ int scan_w_at(int row, int j) { return row * kScanChunk + ((((j >> 3) ^ row) & 7) << 3) + (j & 7); }
// V^T, [column][token].
__device__ __forceinline__ int scan_v_at(int row, int j) { return row * kScanChunk + ((((j >> 3) ^ (row >> 3)) & 7) << 3) + (j & 7); }
// K^T: key column d lies, of each 32, as column 8 a + 4 t + i in row 16 t + 4 a + i, so that the two tiles of 16 rows that make a lane group's
// four columns each leave it eight neighbours: the state's operand.
__device__ __forceinline__ int scan_k_at(int row, int j) {
  return row * kScanChunk + ((((j >> 3) ^ ((row >> 1) & 2) ^ ((row << 1) & 4)) & 7) << 3) + (j & 7);
}
__device__ __forceinline__ int scan_k_row(int d) { return (d & ~31) | ((d & 4) << 2) | ((d & 24) >> 1) | (d & 3); }

// Rows of DP numbers in LDS, a token each, their 16-byte pieces turned by the row so that sixteen rows' lie in different banks.
template <int DP>
__device__ __forceinline__ int scan_row_at(int row, int piece) { return row * DP + 8 * (piece ^ (DP % 128 == 0 ? 2 * (row & 7) : row & 7)); }

// The inclusive sums of la over the wavefront's 64 tokens, 64-bit.
__device__ __forceinline__ double scan_sums(double v) {
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const double u = __shfl_up(v, o, kWave);
    if (lane >= o) v += u;
  }
  return v;
}

// What a chunk's exponents come to, in LDS; exponents of two, so that a weight is a subtraction, a conversion and the hardware's exponential.
struct ScanSums {
  double cum[kScanChunk];                             // c log2(e)
  float keep[kScanChunk];                             // e^(c_n - c_j) b_j
  float b[kScanChunk];                                // b_j times the queries' scale
  float from[kScanChunk];                             // e^(c_i) times the queries' scale
  float decay;                                        // e^(c_n)
  double total;                                       // c_n log2(e)
};
__device__ __forceinline__ float scan_exp2(double x) { return __builtin_amdgcn_exp2f((float)x); }

// A workgroup walks a segment of four chunks with four tiles of 16 columns of a head's state, a wavefront each, in registers: lane (g, r)
// holds column r of rows 32 ks + 8 g + 4 t + i, which is as an operand of q S wants it.  OUT: the segment's outputs, from the state in front of it (the
// slot's where the sequence is one segment, else `work`), and behind the last segment the state into the slot.  Else: the segments' U, but
// the last's, into work [segment][head][column][row], their decays into segment_decay.  Grid (heads, parts of 64 columns, listed sequences x most segments).
//
// What bounds it is the number of a wavefront's instructions, some five cycles each: so the values are scaled and split in two in registers
// (the keys would be twice as many, through LDS), and a segment's exponents are made at once, a chunk a wavefront; with two workgroups a compute unit they wait
// for LDS and each other half of the time, and three would need 168 registers (74 spilled: 48 us where this takes 45).  States
// move through memory twice for every segment where a state a chunk, by kernels of their own, moved four times for every 64 tokens.  The three
// launches, us, before / now: 64 heads of 128 x 64, three sequences of 2,038 tokens 122 / 85, 2,048 tokens 101 / 67, 8,192 419 / 211, 100 29 / 17; 8 of
// 128 x 256 and their sums of keys, 2,038 83 / 60, 2,048 57 / 57, 700 41 / 38, four of 400 57 / 59.
template <int DP, bool OUT>
__global__ __launch_bounds__(kScanThreads, DP <= 128 ? 2 : 1) void scan_walk_kernel(ScanArgs<bf16> a, const int* __restrict__ seq_ids, float* __restrict__ work,
                                                                   float* __restrict__ segment_decay, int max_segments) {
  constexpr int KS = DP / 32, NU = DP / 64, NQ = OUT ? DP / 32 : 1;
  static_assert(kScanMostChunks == kScanThreads / kWave, "a wavefront makes a chunk's exponents");
  extern __shared__ __align__(16) unsigned char scan_lds[];
  __shared__ ScanSums sums[kScanMostChunks];
  const int h = blockIdx.x, z = blockIdx.z / max_segments, sj = blockIdx.z % max_segments;
  const int seq = seq_ids[z];
  const int seq0 = a.cu_q[seq], seq1 = a.cu_q[seq + 1], slot = a.slots[seq];
  const ScanSegments cut(seq1 - seq0, a.heads * gridDim.y);
  const int segments = cut.count, length = cut.each * kScanChunk;
  if (slot < 0 || sj >= segments - (OUT ? 0 : 1)) return;           // the same for the whole workgroup
  const int row_begin = seq0 + sj * length, row_end = row_begin + length < seq1 ? row_begin + length : seq1;
  const size_t idx = scan_segment_index(seq0, z, sj);
  const int tiles = (a.vdim + (a.n ? 1 : 0) + 15) / 16, dpad = (a.dim + 31) / 32 * 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, g = lane / 16, r = lane % 16;
  const int c0 = 64 * blockIdx.y, e = c0 + 16 * wave + r;           // the workgroup's first column, this lane's
  const bool on = c0 + 16 * wave < 16 * tiles, is_n = e == a.vdim && a.n;
  bf16* vt = reinterpret_cast<bf16*>(scan_lds);                     // [column][token]
  bf16* kt = vt + kScanChunk * kScanChunk;                          // [scan_k_row][token]
  bf16* qs = kt + DP * kScanChunk;                                  // [token][DP]
  bf16* wh = qs + kScanChunk * DP;                                  // [query][key]
  bf16* wl = wh + kScanChunk * kScanChunk;

  // a chunk on its way: of K and V units of two tokens x 8 columns, of Q pieces, and this wavefront's 16 keys as an operand
  const size_t qk = (size_t)(h / a.group) * a.dim;
  bf16x8 kx[NU][2], vx[2], qx[NQ], kf[KS];
  auto ask = [&](int row0, int thread) {
    const int n = row_end - row0 < kScanChunk ? row_end - row0 : kScanChunk;
    const bf16 *kp = a.p + (size_t)row0 * a.ld + a.k_off + qk, *qp = a.p + (size_t)row0 * a.ld + a.q_off + qk;
    const bf16* vp = a.p + (size_t)row0 * a.ld + a.v_off + (size_t)h * a.vdim;
    auto token = [&](int j) { return (unsigned)(j < n ? j : n - 1) * (unsigned)a.ld; };   // no load under a condition: what does not exist is not used
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int i = u * kScanThreads + thread, d = 8 * (i % (DP / 8)), j = 2 * (i / (DP / 8));
#pragma unroll
      for (int k = 0; k < 2; ++k) kx[u][k] = *reinterpret_cast<const bf16x8*>(kp + (token(j + k) + (unsigned)(d < a.dim ? d : 0)));
    }
    const int vc = c0 + 8 * (thread % 8);
#pragma unroll
    for (int k = 0; k < 2; ++k) vx[k] = *reinterpret_cast<const bf16x8*>(vp + (token(2 * (thread / 8) + k) + (unsigned)(vc + 8 <= a.vdim ? vc : 0)));
    if (OUT) {
#pragma unroll
      for (int u = 0; u < NQ; ++u) {
        const int i = u * kScanThreads + thread, d = 8 * (i % (DP / 8));
        qx[u] = *reinterpret_cast<const bf16x8*>(qp + (token(i / (DP / 8)) + (unsigned)(d < a.dim ? d : 0)));
      }
      const unsigned own = token(16 * wave + thread % 16);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d = 32 * ks + 8 * (thread % kWave / 16);
        kf[ks] = *reinterpret_cast<const bf16x8*>(kp + (own + (unsigned)(d < a.dim ? d : 0)));
      }
    }
  };
  {
    // a chunk's exponents a wavefront
    const int row0 = row_begin + wave * kScanChunk, n = row_end - row0 < kScanChunk ? row_end - row0 : kScanChunk;   // (none: n is not above 0)
    const bool in = lane < n;
    const size_t at = (size_t)(in ? row0 + lane : row_begin) * a.heads + h;
    const float la = a.la[at], b = a.b[at];
    ask(row_begin, threadIdx.x);
    const double c = scan_sums(in ? (double)la * 1.4426950408889634 : 0.0), total = __shfl(c, kWave - 1, kWave);
    ScanSums& to = sums[wave];
    to.cum[lane] = c;
    to.keep[lane] = in ? scan_exp2(total - c) * b : 0.f;
    to.b[lane] = in ? b * a.q_scale : 0.f;
    to.from[lane] = scan_exp2(c) * a.q_scale;
    if (lane == 0) to.decay = scan_exp2(total), to.total = total;
  }
  // the state in front of the segment
  f32x4 S[KS][2];
  const float* from = work + (idx * a.heads + h) * (size_t)(16 * tiles) * dpad + (size_t)(on ? e : 0) * dpad;
  float* const state = is_n ? a.n + ((size_t)slot * a.heads + h) * a.dim : a.s + ((size_t)slot * a.heads + h) * a.dim * a.vdim + (e < a.vdim ? e : 0);
  const unsigned state_step = is_n ? 1 : a.vdim;
  const bool real = on && (e < a.vdim || is_n);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int d = 32 * ks + 8 * g + 4 * t;
      f32x4 v{0.f, 0.f, 0.f, 0.f};
      if (OUT && segments > 1) {
        v = *reinterpret_cast<const f32x4*>(from + (d < dpad ? d : 0));
      } else if (OUT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = state[(unsigned)(d + i < a.dim ? d + i : 0) * state_step];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) S[ks][t][i] = OUT && on && (segments > 1 ? d < dpad : real && d + i < a.dim) ? v[i] : 0.f;
    }
  // where a thread's pairs of tokens go: the columns k and k + 4 of its eight 16 rows apart, k + 2 turned the other way
  int k_to0[NU], k_to1[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int i = u * kScanThreads + (int)threadIdx.x, d = 8 * (i % (DP / 8)), j = 2 * (i / (DP / 8));
    k_to0[u] = scan_k_at(scan_k_row(d), j), k_to1[u] = scan_k_at(scan_k_row(d + 2), j);
  }
  const int v_to = scan_v_at(8 * ((int)threadIdx.x % 8), 2 * ((int)threadIdx.x / 8));
  const int q_to = scan_row_at<DP>((int)threadIdx.x / (DP / 8), (int)threadIdx.x % (DP / 8));   // (the pieces' rows are whole turns apart)
  static_assert(kScanThreads / (DP / 8) % 8 == 0, "whole turns");
  __syncthreads();
  int at = 0;
  for (int row0 = row_begin; row0 < row_end; row0 += kScanChunk, ++at) {
    const int n = row_end - row0 < kScanChunk ? row_end - row0 : kScanChunk;
    const ScanSums& now = sums[at];
    // (places in LDS and in rows are made anew for every chunk: kept for all of them they would take more registers than there are)
    int thread = threadIdx.x;
    asm volatile("" : "+v"(thread));
    const int lane = thread % kWave, g = lane / 16, r = lane % 16, e = c0 + 16 * wave + r;
    // into LDS: K, V and Q; tokens behind the chunk's end and columns behind the width are zeros
    if (n < kScanChunk || a.dim < DP) {
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int i = u * kScanThreads + (int)threadIdx.x, d = 8 * (i % (DP / 8)), j = 2 * (i / (DP / 8));
#pragma unroll
        for (int k = 0; k < 2; ++k) kx[u][k] = d < a.dim && j + k < n ? kx[u][k] : zero8();
      }
#pragma unroll
      for (int u = 0; u < NQ && OUT; ++u) qx[u] = 8 * ((u * kScanThreads + (int)threadIdx.x) % (DP / 8)) < a.dim ? qx[u] : zero8();
    }
    if (n < kScanChunk || c0 + 64 > a.vdim) {
      const int j = 2 * ((int)threadIdx.x / 8), c = c0 + 8 * ((int)threadIdx.x % 8);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        vx[k] = c + 8 <= a.vdim && j + k < n ? vx[k] : zero8();
        if (a.n && c == a.vdim && j + k < n) vx[k][0] = (bf16)1.f;
      }
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int k = 0; k < 8; ++k)
        *reinterpret_cast<bf16x2*>(kt + (k & 2 ? k_to1[u] : k_to0[u]) + (scan_k_row(k) - (k & 2)) * kScanChunk) = bf16x2{kx[u][0][k], kx[u][1][k]};
#pragma unroll
    for (int k = 0; k < 8; ++k) *reinterpret_cast<bf16x2*>(vt + v_to + k * kScanChunk) = bf16x2{vx[0][k], vx[1][k]};
    if (OUT) {
#pragma unroll
      for (int u = 0; u < NQ; ++u) *reinterpret_cast<bf16x8*>(qs + q_to + u * (kScanThreads / (DP / 8)) * DP) = qx[u];
    }
    __syncthreads();
    f32x4 acc[4];
    if (OUT) {
      // q k of this wavefront's 16 keys, and q S of its 16 columns
      f32x4 x[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) x[it] = acc[it] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        bf16x8 sh, sl;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float s = S[ks][i / 4][i % 4];
          sh[i] = (bf16)s;
          sl[i] = (bf16)(s - (float)sh[i]);
        }
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const bf16x8 q = *reinterpret_cast<const bf16x8*>(qs + scan_row_at<DP>(16 * it + r, 4 * ks + g));
          acc[it] = mfma16(q, sl, acc[it]);
          x[it] = mfma16(kf[ks], q, x[it]);
          acc[it] = mfma16(q, sh, acc[it]);
        }
        if (ks % 2) __builtin_amdgcn_sched_barrier(0);              // (all operands at once would not fit the registers)
      }
      // the weights: on the diagonal from the difference of two sums, elsewhere through the end of the keys' tile, both factors at most one
      const int j0 = 16 * wave + 4 * g;
      const double end = now.cum[16 * wave + 15];
      const f32x4 bj = *reinterpret_cast<const f32x4*>(&now.b[j0]);
      double cj[4];
      float ek[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        cj[k] = now.cum[j0 + k];
        ek[k] = scan_exp2(end - cj[k]) * bj[k];
      }
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        if (it + 1 < wave || (it < wave && wave % 2 == 0)) continue;   // keys behind the queries, but beside the diagonal in the same 32: zeros
        const int i = 16 * it + r;
        const double ci = now.cum[i];
        f32x4 y;
        if (it > wave) {
          const float across = scan_exp2(ci - end);
#pragma unroll
          for (int k = 0; k < 4; ++k) y[k] = x[it][k] * (across * ek[k]);
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) y[k] = it == wave && j0 + k <= i ? x[it][k] * (scan_exp2(ci - cj[k]) * bj[k]) : 0.f;
        }
        bf16x4 hi, lo;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          hi[k] = (bf16)y[k];
          lo[k] = (bf16)(y[k] - (float)hi[k]);
        }
        *reinterpret_cast<bf16x4*>(wh + scan_w_at(i, j0)) = hi;
        *reinterpret_cast<bf16x4*>(wl + scan_w_at(i, j0)) = lo;
      }
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const f32x4 f = *reinterpret_cast<const f32x4*>(&now.from[16 * it + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[it][i] *= f[i];
      }
    }
    if (row0 + kScanChunk < row_end) ask(row0 + kScanChunk, thread);
    bf16x8 v[2];
    if (on) {
#pragma unroll
      for (int k = 0; k < 2; ++k) v[k] = *reinterpret_cast<const bf16x8*>(vt + scan_v_at(16 * wave + r, 32 * k + 8 * g));
      // the values scaled, as the sum of two
      bf16x8 vh[2], vl[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const f32x4 f0 = *reinterpret_cast<const f32x4*>(&now.keep[32 * k + 8 * g]), f1 = *reinterpret_cast<const f32x4*>(&now.keep[32 * k + 8 * g + 4]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float x = (float)v[k][i] * (i < 4 ? f0[i % 4] : f1[i % 4]);
          vh[k][i] = (bf16)x;
          vl[k][i] = (bf16)(x - (float)vh[k][i]);
        }
      }
      const float decay = now.decay;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int row = 32 * ks + 16 * t + r;
          const bf16x8 k0 = *reinterpret_cast<const bf16x8*>(kt + scan_k_at(row, 8 * g)), k1 = *reinterpret_cast<const bf16x8*>(kt + scan_k_at(row, 32 + 8 * g));
          f32x4 u{0.f, 0.f, 0.f, 0.f};
          u = mfma16(k0, vl[0], u);
          u = mfma16(k1, vl[1], u);
          u = mfma16(k0, vh[0], u);
          u = mfma16(k1, vh[1], u);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[ks][t][i] = fmaf(decay, S[ks][t][i], u[i]);
        }
        if (ks % 2) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (OUT) {
      __syncthreads();                                              // every wavefront's weights
      if (on) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int it = 2 * k; it < 4; ++it) {
            acc[it] = mfma16(*reinterpret_cast<const bf16x8*>(wl + scan_w_at(16 * it + r, 32 * k + 8 * g)), v[k], acc[it]);
            acc[it] = mfma16(*reinterpret_cast<const bf16x8*>(wh + scan_w_at(16 * it + r, 32 * k + 8 * g)), v[k], acc[it]);
          }
        if (a.skip && !is_n) {
          const float skip = a.skip[h];
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const bf16x4 x = *reinterpret_cast<const bf16x4*>(vt + scan_v_at(16 * wave + r, 16 * it + 4 * g));
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[it][i] = fmaf(skip, (float)x[i], acc[it][i]);
          }
        }
        // a column of S, or n's
        float *const out = a.out + ((size_t)row0 * a.heads + h) * a.vdim, *const den = a.den + (size_t)row0 * a.heads + h;
        const unsigned step = a.heads * a.vdim, first = 4 * g * step + e;
        if (real && !is_n && n == kScanChunk) {
#pragma unroll
          for (int it = 0; it < 4; ++it)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[first + (16 * it + i) * step] = acc[it][i];
        } else if (real) {
#pragma unroll
          for (int it = 0; it < 4; ++it)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int t = 16 * it + 4 * g + i;
              if (t < n) *(is_n ? den + (unsigned)(t * a.heads) : out + (first + (16 * it + i) * step)) = acc[it][i];
            }
        }
      }
    }
    __syncthreads();                                                // everyone has read this chunk
  }
  if (OUT) {
    if (sj != segments - 1 || !real) return;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = 32 * ks + 8 * g + 4 * t + i;
          if (d < a.dim) state[(unsigned)d * state_step] = S[ks][t][i];
        }
  } else {
    if (on) {
      float* to = work + (idx * a.heads + h) * (size_t)(16 * tiles) * dpad + (size_t)e * dpad;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (32 * ks + 8 * g + 4 * t < dpad) *reinterpret_cast<f32x4*>(to + 32 * ks + 8 * g + 4 * t) = S[ks][t];
    }
    if (threadIdx.x == 0 && blockIdx.y == 0)
      segment_decay[idx * a.heads + h] = scan_exp2(((sums[0].total + sums[1].total) + sums[2].total) + sums[3].total);
  }
}

// Between them: the segments' U become the states in front of them.  A thread an element of a head's state, a batch of segments asked for
// together.  (The state behind the last is scan_walk_kernel's.)
__global__ __launch_bounds__(256) void scan_carry_kernel(ScanArgs<bf16> a, const int* __restrict__ seq_ids, float* __restrict__ work,
                                                         const float* __restrict__ segment_decay) {
  const int z = blockIdx.z, h = blockIdx.y;
  const int seq = seq_ids[z];
  const int row0 = a.cu_q[seq], len = a.cu_q[seq + 1] - row0;
  const int dpad = (a.dim + 31) / 32 * 32, columns = a.vdim + (a.n ? 1 : 0);
  const int slot = a.slots[seq], segments = ScanSegments(len, a.heads * ((columns + 63) / 64)).count;
  if (slot < 0 || segments < 2) return;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= columns * dpad) return;
  const int e = i / dpad, d = i % dpad;
  const size_t size = (size_t)a.heads * ((columns + 15) / 16 * 16) * dpad;
  const size_t first = scan_segment_index(row0, z, 0);
  float* wp = work + first * size + (size_t)h * (size / a.heads) + i;
  const float* dp = segment_decay + first * a.heads + h;
  const bool real = d < a.dim;
  const float* sp = e < a.vdim ? a.s + (((size_t)slot * a.heads + h) * a.dim + (real ? d : 0)) * a.vdim + e
                               : a.n + ((size_t)slot * a.heads + h) * a.dim + (real ? d : 0);
  float S = real ? *sp : 0.f;
  constexpr int kBatch = 8;
  for (int j0 = 0; j0 < segments; j0 += kBatch) {
    float U[kBatch], A[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const int j = j0 + k < segments - 1 ? j0 + k : segments - 2;
      U[k] = wp[(size_t)j * size];
      A[k] = dp[(size_t)j * a.heads];
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k)
      if (j0 + k < segments) {
        wp[(size_t)(j0 + k) * size] = S;
        S = fmaf(A[k], S, U[k]);
      }
  }
}

static int scan_check(const char* what, int nseq, int tokens, int heads, int group, int dim, int vdim, long ld, int q_off, int k_off,
                      int v_off, const void* n, const void* den) {
  PA_REQUIRE(nseq > 0 && nseq <= 65535 && tokens > 0 && heads > 0 && heads <= 65535 && group > 0 && heads % group == 0 && vdim > 0,
             "%s: bad sizes seqs=%d tokens=%d heads=%d (groups of %d) vdim=%d", what, nseq, tokens, heads, group, vdim);
  PA_REQUIRE(dim > 0 && dim <= 256, "%s: a key width of %d is outside 1..256", what, dim);
  PA_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && q_off + (long)(heads / group) * dim <= ld &&
             k_off + (long)(heads / group) * dim <= ld && v_off + (long)heads * vdim <= ld, "%s: the columns do not fit the row of %ld", what, ld);
  PA_REQUIRE((n == nullptr) == (den == nullptr), "%s: a sum of keys and its product with the queries go together", what);
  return 0;
}

}  // namespace pa

using namespace pa;

extern "C" int pa_ssd_gates(void* stream, int dtype, const void* p, long ld, int off, const float* bias, const float* a_log, float* la,
                            float* b, int tokens, int heads) {
  if (tokens == 0) return 0;
  PA_REQUIRE(tokens > 0 && heads > 0 && off >= 0 && off + (long)heads <= ld, "ssd_gates: bad sizes tokens=%d heads=%d", tokens, heads);
  const size_t total = (size_t)tokens * heads;
  const dim3 grid((unsigned)((total + 255) / 256));
  hipStream_t st = (hipStream_t)stream;
  if (dtype == kF32)
    hipLaunchKernelGGL(ssd_gates_kernel<float>, grid, dim3(256), 0, st, (const float*)p, (size_t)ld, off, bias, a_log, la, b, total, heads);
  else if (dtype == kBF16)
    hipLaunchKernelGGL(ssd_gates_kernel<bf16>, grid, dim3(256), 0, st, (const bf16*)p, (size_t)ld, off, bias, a_log, la, b, total, heads);
  else
    return pa::fail("ssd_gates: unknown element type code %d", dtype);
  return check_launch("ssd_gates");
}

// copies of the running maximum: one per column tile of the step kernel, n's included
extern "C" int pa_mlstm_max_copies(int vdim) { return (vdim + kScanCols - 1) / kScanCols + 1; }

extern "C" int pa_mlstm_gates(void* stream, int dtype, const void* p, long ld, int i_off, int f_off, const float* i_bias,
                              const float* f_bias, float cap, float* m, const int* state_slots, const int* cu_q, float* la, float* b,
                              float* floor_out, int nseq, int heads, int vdim, int min_len) {
  if (nseq == 0) return 0;
  PA_REQUIRE(nseq > 0 && nseq <= 65535 && heads > 0 && cap > 0.f && i_off >= 0 && f_off >= 0 && i_off + (long)heads <= ld &&
             f_off + (long)heads <= ld, "mlstm_gates: bad sizes seqs=%d heads=%d cap=%g", nseq, heads, (double)cap);
  hipStream_t st = (hipStream_t)stream;
  const int copies = pa_mlstm_max_copies(vdim);
  if (dtype == kF32)
    hipLaunchKernelGGL(mlstm_gates_kernel<float>, dim3(heads, nseq), dim3(kGateThreads), 0, st, (const float*)p, (size_t)ld, i_off, f_off, i_bias,
                       f_bias, cap, m, copies, state_slots, cu_q, la, b, floor_out, heads, min_len);
  else if (dtype == kBF16)
    hipLaunchKernelGGL(mlstm_gates_kernel<bf16>, dim3(heads, nseq), dim3(kGateThreads), 0, st, (const bf16*)p, (size_t)ld, i_off, f_off, i_bias,
                       f_bias, cap, m, copies, state_slots, cu_q, la, b, floor_out, heads, min_len);
  else
    return pa::fail("mlstm_gates: unknown element type code %d", dtype);
  return check_launch("mlstm_gates");
}

extern "C" int pa_decay_scan(void* stream, int dtype, const void* p, long ld, int q_off, int k_off, int v_off, const float* la,
                             const float* b, float* s, float* n, const float* skip, float q_scale, const int* state_slots,
                             const int* cu_q, float* out, float* den, int nseq, int tokens, int heads, int group, int dim, int vdim,
                             int min_len) {
  if (nseq == 0 || tokens == 0) return 0;
  if (int rc = scan_check("decay_scan", nseq, tokens, heads, group, dim, vdim, ld, q_off, k_off, v_off, n, den)) return rc;
  const dim3 grid((vdim + kScanCols - 1) / kScanCols + (n ? 1 : 0), heads, nseq);
  hipStream_t st = (hipStream_t)stream;
#define PA_SCAN(T, R)                                                                                                         \
  hipLaunchKernelGGL((decay_scan_kernel<T, R>), grid, dim3(kScanThreads), 0, st,                                              \
                     (ScanArgs<T>{(const T*)p, (size_t)ld, q_off, k_off, v_off, heads, group, dim, vdim, la, b, s, n, skip, q_scale, \
                                  state_slots, cu_q, out, den}), min_len)
#define PA_SCAN_R(T)                     \
  do {                                   \
    if (dim <= 32) PA_SCAN(T, 8);        \
    else if (dim <= 64) PA_SCAN(T, 16);  \
    else if (dim <= 128) PA_SCAN(T, 32); \
    else PA_SCAN(T, 64);                 \
  } while (0)
  if (dtype == kF32) PA_SCAN_R(float);
  else if (dtype == kBF16) PA_SCAN_R(bf16);
  else return pa::fail("decay_scan: unknown element type code %d", dtype);
#undef PA_SCAN_R
#undef PA_SCAN
  return check_launch("decay_scan");
}

// a_log given: ssd gates (z_off, bias); else mlstm gates (z_off / bias of i, f_off / f_bias, cap, m, floor_out).
extern "C" int pa_decay_scan_step(void* stream, int dtype, const void* p, long ld, int q_off, int k_off, int v_off, const void* z, long z_ld,
                                  int z_off, int f_off, const float* bias, const float* f_bias, const float* a_log, float cap, float* m, float* floor_out,
                                  float* s, float* n, const float* skip, float q_scale, const int* state_slots, const int* cu_q,
                                  float* out, float* den, int nseq, int heads, int group, int dim, int vdim) {
  if (nseq == 0) return 0;
  if (int rc = scan_check("decay_scan_step", nseq, nseq, heads, group, dim, vdim, ld, q_off, k_off, v_off, n, den)) return rc;
  const bool mlstm = a_log == nullptr;
  PA_REQUIRE(z && z_off >= 0 && z_off + (long)heads <= z_ld && bias && (!mlstm || (f_off >= 0 && f_off + (long)heads <= z_ld && f_bias && cap > 0.f && m &&
             floor_out && n)), "decay_scan_step: a gate's columns do not fit the row of %ld, or a tensor is missing", z_ld);
  const dim3 grid((vdim + kScanCols - 1) / kScanCols + (n ? 1 : 0), heads, nseq);
  hipStream_t st = (hipStream_t)stream;
  const auto launch = [&](auto* kernel, auto zero) {
    typedef decltype(zero) T;
    hipLaunchKernelGGL(kernel, grid, dim3(kScanThreads), 0, st,
                       (ScanArgs<T>{(const T*)p, (size_t)ld, q_off, k_off, v_off, heads, group, dim, vdim, nullptr, nullptr, s, n, skip,
                                    q_scale, state_slots, cu_q, out, den}),
                       (StepGates<T>{(const T*)z, (size_t)z_ld, z_off, f_off, bias, f_bias, a_log, cap, m, pa_mlstm_max_copies(vdim), floor_out}));
  };
  // With a state of 256 rows the kernel of whole quarters has a compute unit to itself by its registers, and of the other three fit:
  // from two workgroups a compute unit to three that one is done in a round.  mLSTM heads of 256 x 512, whole quarters against not: 504
  // workgroups 14.9 / 15.0 us, 576 18.5 / 16.5, 648 21.2 / 19.2, 720 22.5 / 22.2, 792 25.4 / 27.3, 1,728 44.0 / 46.1; 64 columns, 512 14.9
  // / 16.3, 576 20.8 / 18.4, 704 24.0 / 22.2, 768 26.4 / 24.3, 896 28.9 / 30.8.
  const long groups = (long)grid.x * heads * nseq;
  const bool three_fit = dim == 256 && groups > 512 && groups <= 768;
#define PA_STEP(T, R, M)                                                                      \
  do {                                                                                        \
    if (dim == 4 * R && !three_fit) launch(&decay_scan_step_kernel<T, R, M, true>, T(0.f));   \
    else launch(&decay_scan_step_kernel<T, R, M, false>, T(0.f));                             \
  } while (0)
#define PA_STEP_R(T, M)                     \
  do {                                      \
    if (dim <= 32) PA_STEP(T, 8, M);        \
    else if (dim <= 64) PA_STEP(T, 16, M);  \
    else if (dim <= 128) PA_STEP(T, 32, M); \
    else PA_STEP(T, 64, M);                 \
  } while (0)
#define PA_STEP_M(T)                  \
  do {                                \
    if (mlstm) PA_STEP_R(T, true);    \
    else PA_STEP_R(T, false);         \
  } while (0)
  if (dtype == kF32) PA_STEP_M(float);
  else if (dtype == kBF16) PA_STEP_M(bf16);
  else return pa::fail("decay_scan_step: unknown element type code %d", dtype);
#undef PA_STEP_M
#undef PA_STEP_R
#undef PA_STEP
  return check_launch("decay_scan_step");
}

extern "C" int pa_decay_scan_chunked_supports(const void* p, long ld, int q_off, int k_off, int v_off, int dim, int vdim) {
  return dim > 0 && dim <= 256 && dim % 8 == 0 && vdim > 0 && vdim % 8 == 0 && ld % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 &&
         v_off % 8 == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// 32-bit words of workspace: the segments' states, then their decays
extern "C" long pa_decay_scan_chunked_workspace(int nlisted, int tokens, int heads, int dim, int vdim, int with_n) {
  const long tiles = (vdim + (with_n ? 1 : 0) + 15) / 16, dpad = (dim + 31) / 32 * 32;
  return ((long)tokens / kScanChunk + nlisted) * heads * (tiles * 16 * dpad + 1);
}

// The listed sequences (at most max_len tokens each), bfloat16.
extern "C" int pa_decay_scan_chunked(void* stream, const void* p, long ld, int q_off, int k_off, int v_off, const float* la, const float* b,
                                     float* s, float* n, const float* skip, float q_scale, const int* state_slots, const int* cu_q,
                                     const int* seq_ids, float* out, float* den, float* work, int nlisted, int tokens, int max_len,
                                     int heads, int group, int dim, int vdim) {
  if (nlisted == 0 || tokens == 0 || max_len == 0) return 0;
  if (int rc = scan_check("decay_scan_chunked", nlisted, tokens, heads, group, dim, vdim, ld, q_off, k_off, v_off, n, den)) return rc;
  PA_REQUIRE(pa_decay_scan_chunked_supports(p, ld, q_off, k_off, v_off, dim, vdim), "decay_scan_chunked: widths %d and %d, or columns that "
             "are no whole 16-byte pieces", dim, vdim);
  PA_REQUIRE(seq_ids && work, "decay_scan_chunked: no list of sequences or no workspace");
  const int max_chunks = (max_len + kScanChunk - 1) / kScanChunk;
  PA_REQUIRE((long)nlisted * max_chunks <= 65535, "decay_scan_chunked: %d sequences x %d chunks exceed the grid", nlisted, max_chunks);
  const ScanArgs<bf16> a{(const bf16*)p, (size_t)ld, q_off, k_off, v_off, heads, group, dim, vdim, la, b, s, n, skip, q_scale, state_slots,
                         cu_q, out, den};
  const int tiles = (vdim + (n ? 1 : 0) + 15) / 16, dpad = (dim + 31) / 32 * 32, columns = vdim + (n ? 1 : 0);
  int max_segments = 1;                                             // of any length up to the longest
  for (int c = 1; c <= max_chunks; ++c) {
    const int count = ScanSegments(c * kScanChunk, heads * ((tiles + 3) / 4)).count;
    max_segments = count > max_segments ? count : max_segments;
  }
  const dim3 grid(heads, (tiles + 3) / 4, nlisted * max_segments);
  float* segment_decay = work + ((long)tokens / kScanChunk + nlisted) * heads * (long)(tiles * 16) * dpad;
  hipStream_t st = (hipStream_t)stream;
#define PA_CHUNKED(DP)                                                                                                          \
  do {                                                                                                                          \
    constexpr int lds_state = (kScanChunk + DP) * kScanChunk * (int)sizeof(bf16), lds_all = lds_state + (DP + 2 * kScanChunk) * kScanChunk * (int)sizeof(bf16); \
    static const hipError_t allowed = [] {                                                                                      \
      const hipError_t one = hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_walk_kernel<DP, true>),                    \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds_all);                          \
      return one != hipSuccess ? one : hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_walk_kernel<DP, false>),         \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds_state);              \
    }();                                                                                                                        \
    PA_REQUIRE(allowed == hipSuccess, "decay_scan_chunked: %d bytes of LDS refused: %s", lds_all, hipGetErrorString(allowed));      \
    if (max_segments > 1) {                                                                                                     \
      hipLaunchKernelGGL((scan_walk_kernel<DP, false>), grid, dim3(kScanThreads), lds_state, st, a, seq_ids, work, segment_decay, max_segments); \
      hipLaunchKernelGGL(scan_carry_kernel, dim3((columns * dpad + 255) / 256, heads, nlisted), dim3(256), 0, st, a, seq_ids, work, \
                         segment_decay);                                                                                        \
    }                                                                                                                           \
    hipLaunchKernelGGL((scan_walk_kernel<DP, true>), grid, dim3(kScanThreads), lds_all, st, a, seq_ids, work, segment_decay, max_segments); \
  } while (0)
  if (dim <= 64) PA_CHUNKED(64);
  else if (dim <= 128) PA_CHUNKED(128);
  else PA_CHUNKED(256);
#undef PA_CHUNKED
  return check_launch("decay_scan_chunked");
}
