// Eight neighbouring elements of a row that a row-wise kernel adds to its stream, asked for apart from being used: a row is a
// workgroup, what bounds such a kernel is one thread's path, and a load that is converted or added where it stands is a trip to
// memory of its own.
#pragma once
#include <type_traits>

#include "common.h"

namespace pa {

enum RowFrom : int { kRowNone = 0, kRowTensor = 1, kRowSlices = 2 };   // nothing, a tensor, `slices` 32-bit partial sums added in order

struct Eight32 {
  f32x4 v[2];
  __device__ __forceinline__ void ask(const float* p) {
    v[0] = *reinterpret_cast<const f32x4*>(p);
    v[1] = *reinterpret_cast<const f32x4*>(p + 4);
  }
  __device__ __forceinline__ float operator[](int i) const { return v[i / 4][i % 4]; }
};
template <typename T> struct EightOf;
template <> struct EightOf<float> : Eight32 {};
template <> struct EightOf<bf16> {
  bf16x8 v;
  __device__ __forceinline__ void ask(const bf16* p) { v = *reinterpret_cast<const bf16x8*>(p); }
  __device__ __forceinline__ float operator[](int i) const { return (float)v[i]; }
};

// How many partial sums a thread asks for together, 1, 2 or 4 and at most MOST (a thread of several pieces keeps its registers):
// launch(the number, as a type).  Three and more come four at a time; exact numbers would be kernels of their own for a load of the L1.
template <int MOST, typename Launch>
inline void by_slices_at_once(bool together, int slices, Launch launch) {
  const int n = !together || slices <= 1 ? 1 : slices == 2 ? 2 : 4;
  if constexpr (MOST >= 4) {
    if (n == 4) return launch(std::integral_constant<int, 4>());
  }
  if constexpr (MOST >= 2) {
    if (n >= 2) return launch(std::integral_constant<int, 2>());
  }
  launch(std::integral_constant<int, 1>());
}
// The norms of one row a workgroup ask for partial sums together up to so many elements, where a thread's trips to memory are what they
// take; more are bound by memory, which serves one slice after the other as fast or faster (pieces of slices whose distance is a power
// of two lie in the same channel).  us, two or four together / one at a time: [150, 1024] behind four 3.16 / 3.65, [512, 1024] 4.19 /
// 4.45 and behind six 5.57 / 6.34, [700, 1024] 6.67 / 7.23, [256, 2560] 6.49 / 7.17, but [300, 2560] 8.08 / 7.86, [300, 4096] 11.1 / 9.8,
// [700, 2560] 12.9 / 12.0, [1000, 1024] level; in front of a 32-bit stream [256, 2048] behind four 4.62 / 5.23, [700, 2048] 9.73 / 9.38,
// [2048, 2048] behind eight 36.9 / 34.1.
inline bool sums_together(int nrows, int hidden) { return (long)nrows * hidden <= 720000; }

// The VPT pieces of a thread.  AT_ONCE: partial sums of each asked for together.
template <typename T, int FROM, int AT_ONCE, int VPT>
struct RowPieces {
  EightOf<T> y[VPT];
  Eight32 part[VPT][AT_ONCE];

  // slices that are not there: the one asked for first, again
  __device__ __forceinline__ void ask_slices(int v, const float* parts, int slices, size_t stride, size_t at, int first) {
#pragma unroll
    for (int q = 0; q < AT_ONCE; ++q) part[v][q].ask(parts + (size_t)(first + q < slices ? first + q : first) * stride + at);
  }
  __device__ __forceinline__ void ask(int v, const T* tensor, const float* parts, int slices, size_t stride, size_t at) {
    if constexpr (FROM == kRowTensor) y[v].ask(tensor + at);
    if constexpr (FROM == kRowSlices) ask_slices(v, parts, slices, stride, at, 0);
  }
  // Behind everything that is asked for before it is waited for.
  __device__ __forceinline__ void have() const {
    if constexpr (FROM == kRowSlices) {
#pragma unroll
      for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int q = 0; q < AT_ONCE; ++q) arrived(part[v][q].v[0]), arrived(part[v][q].v[1]);
    }
  }
  // The pieces' elements, piece v's at row + at[v].
  __device__ __forceinline__ void take(float (&out)[VPT][8], const float* parts, int slices, size_t stride, size_t row,
                                       const int (&at)[VPT]) {
    if constexpr (FROM == kRowTensor) {
#pragma unroll
      for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int i = 0; i < 8; ++i) out[v][i] = y[v][i];
    }
    if constexpr (FROM == kRowSlices) {
      for (int first = 0; first < slices; first += AT_ONCE) {
        if (first) {
#pragma unroll
          for (int v = 0; v < VPT; ++v) ask_slices(v, parts, slices, stride, row + at[v], first);
          have();
        }
#pragma unroll
        for (int q = 0; q < AT_ONCE; ++q) {
          if (first + q >= slices) break;
#pragma unroll
          for (int v = 0; v < VPT; ++v)
#pragma unroll
            for (int i = 0; i < 8; ++i) out[v][i] = first + q ? out[v][i] + part[v][q][i] : part[v][q][i];
        }
      }
    }
  }
};

}  // namespace pa
