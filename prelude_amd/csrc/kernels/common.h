// Shared device helpers for the gfx950 kernels: element types, conversions,
// wavefront (64 lanes) and block reductions, and the host-side error channel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pa {

constexpr int kWave = 64;

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Element type codes shared with the Python side.
enum DType : int { kF32 = 0, kBF16 = 1 };

// The activation of a gated feed-forward act(gate) * up, by a code shared with the Python side: SiLU
// x / (1 + e^-x) (crates/prelude-cuda/src/kernels/kernels_src/common/common.cuh:78-80, what the reference's Qwen3
// is wired to, qwen3.rs:429-447) or GELU in its tanh form 0.5 x (1 + tanh(sqrt(2 / pi) (x + 0.044715 x^3))) (the
// reference's Activation::GeluPytorchTanh, crates/prelude-core/src/models/commons/activation.rs:3-25).  The code
// is the same in every lane, so the choice is a branch, and SiLU's arithmetic is what it was without it.
enum GateActivation : int { kActSilu = 0, kActGeluTanh = 1, kActCount = 2 };
__device__ __forceinline__ float gate_activation(float x, int act) {
  if (act == kActGeluTanh) return 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
  return x / (1.0f + expf(-x));
}

// A gated pair with both halves clamped: g = min(g, limit), u = clamp(u, -limit, limit), and
// g * sigmoid(alpha * g) * (u + 1); `limit` and `alpha` are the model's constants.
__device__ __forceinline__ float clamped_gate(float g, float u, float limit, float alpha) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
}

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16 v) { return static_cast<float>(v); }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) { return static_cast<bf16>(v); }  // round to nearest even

// sigmoid, SiLU and the gated activations for a result that is rounded to T: behind bfloat16 the hardware's exponential and
// reciprocal serve (a few units of the 24th bit); GELU in its tanh form is x sigmoid(2 u), u = sqrt(2 / pi) (x + 0.044715 x^3).
template <typename T>
__device__ __forceinline__ float sigmoid_of(float z) {
  if (sizeof(T) == 2) return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
  return 1.0f / (1.0f + expf(-z));
}
template <typename T>
__device__ __forceinline__ float silu_of(float z) { return sizeof(T) == 2 ? z * sigmoid_of<T>(z) : z / (1.0f + expf(-z)); }
template <typename T>
__device__ __forceinline__ float gate_activation_of(float z, int act) {
  if (sizeof(T) == 2) return z * sigmoid_of<T>(act == kActGeluTanh ? 1.5957691216057308f * (z + 0.044715f * z * z * z) : z);
  return gate_activation(z, act);
}

// Waits for a load behind those asked for before it.  What is used only under a condition is otherwise loaded there, whatever stands
// between: the compiler moves a load to its one use, past barriers to the scheduler, and waits for it before it asks for the next.
__device__ __forceinline__ void arrived(const f32x4& v) { asm volatile("" ::"v"(v)); }

// Reductions over a wavefront, all 64 lanes at work, the result in every lane: lane l takes its partner's value at l ^ 32, 16, 8, 4, 2
// and 1 in turn.  The exchanges are the vector ALU's own (v_permlane32_swap and 16_swap give a lane its own value and its partner's;
// a rotation by eight or four lanes of a row of sixteen brings the partner's once the row repeats every sixteen or eight lanes):
// an exchange through LDS takes some 100 cycles, six of them in a row were a tenth of a microsecond of every norm's chain.
template <typename Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
  unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  u = __float_as_uint(op(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = op(__uint_as_float(b[0]), __uint_as_float(b[1]));
#define PA_FROM_LANE(CTRL) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true))
  v = op(v, PA_FROM_LANE(0x128));   // row_ror:8
  v = op(v, PA_FROM_LANE(0x124));   // row_ror:4
  v = op(v, PA_FROM_LANE(0x4e));    // quad_perm [2, 3, 0, 1]
  v = op(v, PA_FROM_LANE(0xb1));    // quad_perm [1, 0, 3, 2]
#undef PA_FROM_LANE
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
  return wave_reduce(v, [](float x, float y) { return x + y; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float x, float y) { return fmaxf(x, y); });
}

// The first key the query at `pos` sees: the whole past, a sliding window of `window` places (its own included), or the start
// of its own chunk of `chunk` places, counted from the sequence's start (0: none of that kind).
__device__ __forceinline__ int first_visible(int pos, int window, int chunk) {
  int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  if (chunk > 0) {
    const int c = pos / chunk * chunk;
    lo = c > lo ? c : lo;
  }
  return lo;
}

// Item i of a head's part whose first rot_dims elements turn in pairs (2i, 2i + 1) by p * inv_freq[i]: a turned pair (i below
// rot_dims / 2) or one of the elements behind them as it is; rot_dims / 2 + (width - rot_dims) items a part.
template <typename T>
__device__ __forceinline__ void rotate_part(const T* __restrict__ src, T* __restrict__ dst, int i, float p,
                                            const float* __restrict__ inv_freq, int rot_dims) {
  if (i < rot_dims / 2) {
    float s, c;
    sincosf(p * inv_freq[i], &s, &c);
    const float u = to_f32(src[2 * i]), v = to_f32(src[2 * i + 1]);
    dst[2 * i] = from_f32<T>(u * c - v * s);
    dst[2 * i + 1] = from_f32<T>(v * c + u * s);
  } else {
    const int d = i + rot_dims - rot_dims / 2;
    dst[d] = src[d];
  }
}

// Sum over a block of up to 1024 threads; every thread gets the result.
// `scratch` is LDS for at least 16 floats.  The order of the additions is
// fixed by the thread layout alone, so a row's result never depends on what
// else the launch holds.
// `fresh`: no thread of the block has touched it before (a barrier less).
__device__ __forceinline__ float block_sum(float v, float* scratch, bool fresh = false) {
  v = wave_sum(v);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int nwaves = (blockDim.x + kWave - 1) / kWave;
  if (!fresh) __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nwaves; ++i) t += scratch[i];
  return t;
}

}  // namespace pa

// ---- host side -----------------------------------------------------------
// Every entry point returns 0 on success.  On a refusal (a size the kernel
// does not take, a launch error) it returns nonzero and leaves a message for
// pa_last_error().
extern "C" const char* pa_last_error();
namespace pa {
int fail(const char* fmt, ...);
int check_launch(const char* what);
// Weights that the kernels behind this one stream, read ahead into the L2s by workgroups that a small grid has room for
// while its own wait for memory.  A weight is a row of units, what one workgroup of its product streams (a tile of 16
// rows); unit u is read on the XCD that workgroup u is dealt to, every eighth place, and stays in that XCD's L2.
constexpr int kAheadMost = 4;    // weights
constexpr int kAheadLoads = 8;   // of 16 bytes that a thread has in flight
struct Ahead {
  const char* data[kAheadMost];
  int unit[kAheadMost];    // bytes, a multiple of 16
  int units[kAheadMost];
  int places;              // workgroups that read them, 0: none
};

// How many workgroups of `threads` threads a weight's units take: each has kAheadLoads loads a thread out, of one unit.
__host__ __device__ __forceinline__ int ahead_places(int unit, int units, int threads) {
  const int piece = threads * 16 * kAheadLoads;
  return (units + 7) / 8 * 8 * ((unit + piece - 1) / piece);
}

// The share of workgroup `place`; it lies on XCD place % 8.
__device__ __forceinline__ void read_ahead(const Ahead& a, int place, int threads) {
#pragma unroll
  for (int i = 0; i < kAheadMost; ++i) {
    const int row = (a.units[i] + 7) / 8 * 8, all = ahead_places(a.unit[i], a.units[i], threads);
    if (place >= 0 && place < all && place % row < a.units[i]) {
      const char* p = a.data[i] + (size_t)(place % row) * a.unit[i];
      const int at = (place / row) * threads * 16 * kAheadLoads + threadIdx.x * 16;
      f32x4 v[kAheadLoads];
#pragma unroll
      for (int j = 0; j < kAheadLoads; ++j) {
        const int b = at + j * threads * 16;
        v[j] = *reinterpret_cast<const f32x4*>(p + (b < a.unit[i] ? b : 0));   // past the unit's end: its start again
      }
#pragma unroll
      for (int j = 0; j < kAheadLoads; ++j) asm volatile("" ::"v"(v[j]));   // nothing uses them: keep the loads
    }
    place -= all;
  }
}

}  // namespace pa

#define PA_REQUIRE(cond, ...)                  \
  do {                                         \
    if (!(cond)) return pa::fail(__VA_ARGS__); \
  } while (0)
