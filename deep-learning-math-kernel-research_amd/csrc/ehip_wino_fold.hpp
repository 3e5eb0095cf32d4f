// The output transform of a Winograd tile, value by value (the ring kernels and the kernel that runs a layer whole).
#ifndef EHIP_WINO_FOLD_HPP
#define EHIP_WINO_FOLD_HPP
#include <hip/hip_runtime.h>
#include <utility>

namespace ehip {

namespace {

// Y = At M A one value at a time.  The positions of a tile are visited in the order kOrder of their column, and inside a
// column in the order kOrder of their row, chosen so that the one-dimensional transform (out6_1d, out5_1d) folds a value
// into at most four running ones as it comes: the same operations on the same operands as the whole-column form, which
// needs all A at once.  step k takes the k-th value of the order; after the last, result() holds the A - 2 outputs.
template <int A> struct Fold;
template <> struct Fold<6> {
  static constexpr int kOrder[6] = {1, 2, 3, 4, 0, 5};
  static __device__ __forceinline__ int order(int i) { return (int)((0x504321504321ull >> (4 * i)) & 15u); }   // (i runs on into the next tile)
  template <int K>
  static __device__ __forceinline__ void step(float (&s)[4], float x)
  {
    const float z0 = 1.5f, z1 = 2.25f, z2 = 3.375f, z3 = 0.625f, z4 = 0.390625f, z5 = 0.244140625f;
    if constexpr (K == 0) s[0] = x;
    else if constexpr (K == 1) {
      const float f1 = s[0];
      s[0] = f1 + x;       // t0
      s[1] = f1 - x;       // t2
    } else if constexpr (K == 2) s[2] = x;
    else if constexpr (K == 3) {
      const float t0 = s[0], t2 = s[1], t1 = s[2] + x, t3 = s[2] - x;
      s[0] = t0 + t1;
      s[1] = __builtin_fmaf(t2, z3, t3 * z0);
      s[2] = __builtin_fmaf(t0, z4, t1 * z1);
      s[3] = __builtin_fmaf(t2, z5, t3 * z2);
    } else if constexpr (K == 4) s[0] = s[0] + x;
    else s[3] = s[3] + x;
  }
  // the same steps with every running value updated in its own register (see the column loop)
  template <int K>
  static __device__ __forceinline__ void step_in_place(float (&s)[4], float x)
  {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (K == 0) asm volatile("v_mov_b32 %0, %1" : "+v"(s[0]) : "v"(x));
    else if constexpr (K == 1) asm volatile("v_sub_f32 %1, %0, %2\n\tv_add_f32 %0, %0, %2" : "+v"(s[0]), "+v"(s[1]) : "v"(x));
    else if constexpr (K == 2) asm volatile("v_mov_b32 %0, %1" : "+v"(s[2]) : "v"(x));
    else if constexpr (K == 3) {
      float a, b;
      asm volatile("v_add_f32 %4, %2, %6\n\tv_sub_f32 %5, %2, %6\n\t"
                   "v_mul_f32 %2, %8, %4\n\tv_fma_f32 %2, %0, %11, %2\n\tv_add_f32 %0, %0, %4\n\t"
                   "v_mul_f32 %3, %9, %5\n\tv_fma_f32 %3, %1, %12, %3\n\t"
                   "v_mul_f32 %5, %7, %5\n\tv_fma_f32 %1, %1, %10, %5"
                   : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "=&v"(a), "=&v"(b)
                   : "v"(x), "s"(1.5f), "s"(2.25f), "s"(3.375f), "s"(0.625f), "s"(0.390625f), "s"(0.244140625f));
    } else if constexpr (K == 4) asm volatile("v_add_f32 %0, %0, %1" : "+v"(s[0]) : "v"(x));
    else asm volatile("v_add_f32 %0, %0, %1" : "+v"(s[3]) : "v"(x));
#endif
  }
  static __device__ __forceinline__ float result(const float (&s)[4], int r) { return s[r]; }
};
template <> struct Fold<5> {
  static constexpr int kOrder[5] = {1, 2, 3, 0, 4};
  static __device__ __forceinline__ int order(int i) { return (int)((0x4032140321ull >> (4 * i)) & 15u); }
  template <int K>
  static __device__ __forceinline__ void step(float (&s)[4], float x)
  {
    const float z0 = 0.3333333333333333f, z1 = 0.6666666666666666f, z2 = 1.3333333333333333f;
    if constexpr (K == 0) s[0] = x;
    else if constexpr (K == 1) {
      const float f1 = s[0];
      s[0] = __builtin_fmaf(x, z0, f1);     // t1
      s[1] = __builtin_fmaf(x, z0, -f1);
    } else if constexpr (K == 2) {
      s[1] = __builtin_fmaf(-x, z1, s[1]);
      s[2] = x;
    } else if constexpr (K == 3) s[3] = __builtin_fmaf(s[2], z2, x) + s[0];
    else s[2] = __builtin_fmaf(s[2], z0, x) + s[0];
  }
  template <int K>
  static __device__ __forceinline__ void step_in_place(float (&s)[4], float x)
  {
#if defined(__HIP_DEVICE_COMPILE__)
    const float z0 = 0.3333333333333333f, z1 = 0.6666666666666666f, z2 = 1.3333333333333333f;
    if constexpr (K == 0) asm volatile("v_mov_b32 %0, %1" : "+v"(s[0]) : "v"(x));
    else if constexpr (K == 1)
      asm volatile("v_fma_f32 %1, %2, %3, -%0\n\tv_fma_f32 %0, %2, %3, %0" : "+v"(s[0]), "+v"(s[1]) : "v"(x), "s"(z0));
    else if constexpr (K == 2)
      asm volatile("v_fma_f32 %0, -%2, %3, %0\n\tv_mov_b32 %1, %2" : "+v"(s[1]), "+v"(s[2]) : "v"(x), "s"(z1));
    else if constexpr (K == 3)
      asm volatile("v_fma_f32 %0, %1, %3, %2\n\tv_add_f32 %0, %0, %4" : "+v"(s[3]) : "v"(s[2]), "v"(x), "s"(z2), "v"(s[0]));
    else asm volatile("v_fma_f32 %0, %0, %2, %1\n\tv_add_f32 %0, %0, %3" : "+v"(s[2]) : "v"(x), "s"(z0), "v"(s[0]));
#endif
  }
  static __device__ __forceinline__ float result(const float (&s)[4], int r) { return r == 0 ? s[3] : (r == 1 ? s[1] : s[2]); }
};
template <> struct Fold<4> {   // (a two-dimensional formula in the reference: the positions are kept)
  static constexpr int kOrder[4] = {0, 1, 2, 3};
  static __device__ __forceinline__ int order(int i) { return i & 3; }
};
template <int A, int... K>
__device__ __forceinline__ void fold_step(int k, float (&s)[4], float x, std::integer_sequence<int, K...>)
{
  ((k == K ? Fold<A>::template step<K>(s, x) : (void)0), ...);
}
// the running values that exist after step k stay where they are computed
__device__ __forceinline__ void pin(float (&s)[4], int k)
{
  asm volatile("" : "+v"(s[0]));
  if (k >= 1) asm volatile("" : "+v"(s[1]));
  if (k >= 2) asm volatile("" : "+v"(s[2]));
  if (k >= 3) asm volatile("" : "+v"(s[3]));
}

}  // namespace

}  // namespace ehip
#endif
