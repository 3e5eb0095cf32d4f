// What the kernels that finish a Winograd tile in the lane have in common: one lane holds a tile x four channels, and the
// four lanes of a tile turn their requantized values into whole cells of the output.  (u8 / s8 and f32 output; the
// arithmetic per value is output_tile's, ehip_wino.hip.)
#ifndef EHIP_WINO_PACK_HPP
#define EHIP_WINO_PACK_HPP
#include "ehip_internal.hpp"
#include "ehip_wino_input.hpp"
#include "ehip_wino_tiles.hpp"
#include <type_traits>

namespace ehip {

namespace {

// The pieces of output_tile (ehip_wino.hip) for u8 / s8 output with few registers: one channel at a time, its bytes
// packed into the pixels' dwords as they come (16 dwords live instead of 4 x 16 floats; the old output of the in-place
// sum stays packed as well).  Same operations in the same order per value as output_tile.
// pack_channel: channel k of the lane's four -- bias, output scale, old output, ReLU, rounding, byte k of the dwords.
// (E: pixels, the tile's or one row of it; CLAMP: both bounds of the ReLU explicitly, see below)
template <int OUT, int A, int E = (A - 2) * (A - 2), bool CLAMP = false>
__device__ __forceinline__ void pack_channel(const float *o, float b, int k, bool with_relu, float repS, float z, bool with_sum,
                                             const unsigned *old, unsigned *pk)
{
  static_assert(OUT == EHIP_U8 || OUT == EHIP_S8, "quantized output");
#pragma unroll
  for (int e = 0; e < E; ++e) {
    float r = o[e] + b;
    r = __builtin_fmaf(r, repS, z);
    if (with_sum) {
      const unsigned ob = (old[e] >> (8 * k)) & 0xffu;
      r = r + (OUT == EHIP_U8 ? (float)ob : (float)(int)(signed char)ob);
    }
    if (with_relu) {
      // (v_cvt_pk_u8_f32 itself clamps to 0..255 and makes a NaN 0, all that the ReLU asks for of a u8 code; s8 has its own
      // bound.  The ring kernel keeps both: it has no registers to spare, and without this instruction in the u8 branch the compiler
      // places the values of all branches otherwise, 25 instead of 15 of them in scratch memory with 64 channels x 64 tiles)
      if (OUT == EHIP_S8 || CLAMP) r = __builtin_amdgcn_fmed3f(r, 0.0f, OUT == EHIP_S8 ? 127.0f : 255.0f);
      if (A == 4) r = __builtin_floorf(r);
      pk[e] = __builtin_amdgcn_cvt_pk_u8_f32(r, k, pk[e]);
    } else if (A == 4) {
      const float fl = __builtin_floorf(r);
      if (OUT == EHIP_U8) pk[e] = __builtin_amdgcn_cvt_pk_u8_f32(r >= 0.0f ? fl : 300.0f, k, pk[e]);
      else pk[e] |= ((unsigned)ssat8(cvt_s32_rne(fl)) & 0xffu) << (8 * k);
    } else {
      if (OUT == EHIP_U8) pk[e] = __builtin_amdgcn_cvt_pk_u8_f32(r >= -0.5f ? r : 300.0f, k, pk[e]);
      else pk[e] |= ((unsigned)ssat8(cvt_s32_rne(r)) & 0xffu) << (8 * k);
    }
  }
}

// 4 x 4 transpose of dwords between four registers and the four 16-lane rows of a wave: register j of row g becomes
// register g of row j (v_permlane32_swap exchanges the upper rows of one register with the lower rows of another,
// v_permlane16_swap the odd rows with the even ones).  All lanes take part.
__device__ __forceinline__ void rows_transpose(unsigned &x0, unsigned &x1, unsigned &x2, unsigned &x3)
{
  auto a = __builtin_amdgcn_permlane32_swap(x0, x2, false, false);
  auto b = __builtin_amdgcn_permlane32_swap(x1, x3, false, false);
  auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  x0 = c[0];
  x1 = c[1];
  x2 = d[0];
  x3 = d[1];
}

// Output by whole cells of 16 channels: the four lanes of a tile (rows g = 0 .. 3 of the wave, four channels each) hold
// the 16 bytes of every pixel between them; after the transpose the lane of row g holds the whole cell of the pixel in
// column g of the tile's row i and writes it with one 16-byte store (a wave then covers 16 tiles x 4 pixels of an
// image row = up to 1 KB in one piece, where dword stores leave 16 pieces of 16 bytes per instruction).
// block: the tile's image and channel block; ok: the tile exists.  Called by all lanes.
// (store_row: row i of the tile, pk its M pixels)
template <int A>
__device__ __forceinline__ void store_row(const unsigned *pk, uint8_t *block, int i, int g, bool ok, int th, int tw, int oh_n, int ow_n,
                                          int px)
{
  constexpr int M = A - 2;
  unsigned c0 = pk[0], c1 = pk[1], c2 = M > 2 ? pk[M > 2 ? 2 : 0] : 0u, c3 = M > 3 ? pk[M > 3 ? 3 : 0] : 0u;
  rows_transpose(c0, c1, c2, c3);
  const int oh = M * th + i, ow = M * tw + g;
  if (ok && g < M && oh < oh_n && ow < ow_n) {
    // (non-temporal: the output would only push the transformed input, which the other channel blocks' workgroups
    // still read, out of the L2 -- 128 -> 128 at 112 x 112: 130 -> 100 us)
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const v4u vv = {c0, c1, c2, c3};
    __builtin_nontemporal_store(vv, reinterpret_cast<v4u *>(block + ((size_t)oh * ow_n + ow) * px));
  }
}
template <int A>
__device__ __forceinline__ void store_cells(const unsigned *pk, uint8_t *block, int g, bool ok, int th, int tw, int oh_n, int ow_n,
                                            int px)
{
  constexpr int M = A - 2;
#pragma unroll
  for (int i = 0; i < M; ++i) store_row<A>(pk + M * i, block, i, g, ok, th, tw, oh_n, ow_n, px);
}

// the old output of the in-place sum the same way round: cells in, the lane's four channels of every pixel out
template <int A>
__device__ __forceinline__ void load_old_row(unsigned *old, const uint8_t *block, int i, int g, int th, int tw, int oh_n, int ow_n, int px)
{
  constexpr int M = A - 2;
  const int oh = M * th + i, ow = M * tw + g;
  const bool in = g < M && oh < oh_n && ow < ow_n;
  const uint4 c = *reinterpret_cast<const uint4 *>(block + (in ? ((size_t)oh * ow_n + ow) * px : 0));
  unsigned c0 = c.x, c1 = c.y, c2 = c.z, c3 = c.w;
  rows_transpose(c0, c1, c2, c3);
  old[0] = c0;
  old[1] = c1;
  if (M > 2) old[M > 2 ? 2 : 0] = c2;
  if (M > 3) old[M > 3 ? 3 : 0] = c3;
}
template <int A>
__device__ __forceinline__ void load_old_cells(unsigned *old, const uint8_t *block, int g, int th, int tw, int oh_n, int ow_n, int px)
{
  constexpr int M = A - 2;
#pragma unroll
  for (int i = 0; i < M; ++i) load_old_row<A>(old + M * i, block, i, g, th, tw, oh_n, ow_n, px);
}

// All positions of the lane's tile x four channels -> the output: Y = At M A channel by channel, packed, and written by
// whole cells.  Called by all lanes of the wave (ok: the lane's tile and channels exist).
template <int OUT, int A>
__device__ __forceinline__ void output_tile_packed(const float4 *m, const float4 &bias, bool with_relu, float repS, float z,
                                                   uint8_t *block, int g, bool ok, int th, int tw, int oh_n, int ow_n,
                                                   bool with_sum, int px)
{
  constexpr int AA = A * A, M = A - 2;
  unsigned pk[M * M], old[M * M];
#pragma unroll
  for (int e = 0; e < M * M; ++e) pk[e] = 0u;
  if (with_sum) load_old_cells<A>(old, block, g, th, tw, oh_n, ow_n, px);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float f[AA], o[M * M];
#pragma unroll
    for (int e = 0; e < AA; ++e) f[e] = comp_of(m[e], k);
    wino::tile_output<A>(f, o);
    pack_channel<OUT, A>(o, comp_of(bias, k), k, with_relu, repS, z, with_sum, old, pk);
    // (one channel after the other: interleaved, the four transforms' intermediates do not fit the registers)
    __builtin_amdgcn_sched_barrier(0);
  }
  store_cells<A>(pk, block, g, ok, th, tw, oh_n, ow_n, px);
}

// f32 output (no output scale, no in-place sum here): bias and ReLU as output_tile applies them, and the lane's four
// channels of every pixel leave as one 16-byte store (the four lanes of a tile write the 64 bytes of a pixel's block).
// y: [channel][pixel]; block: the tile's image and channel block, in floats.
template <int A>
__device__ __forceinline__ void finish_channel_f32(float *y, float b, bool with_bias, bool with_relu)
{
  constexpr int M = A - 2;
#pragma unroll
  for (int e = 0; e < M * M; ++e) {
    float r = y[e];
    if (with_bias) r = r + b;
    if (with_relu) r = r > 0.0f ? r : 0.0f;
    y[e] = r;
  }
}
// register j of lane q of every quad of lanes becomes register q of lane j (two exchanges, with lane ^ 1 and lane ^ 2)
__device__ __forceinline__ void quad_transpose4(float &x0, float &x1, float &x2, float &x3, int lane)
{
#if defined(__HIP_DEVICE_COMPILE__)
  const bool odd = (lane & 1) != 0, hi = (lane & 2) != 0;
  auto dpp = [](float v, auto perm) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), decltype(perm)::value, 0xf, 0xf, true));
  };
  const float r01 = dpp(odd ? x0 : x1, std::integral_constant<int, 0xB1>{}), r23 = dpp(odd ? x2 : x3, std::integral_constant<int, 0xB1>{});
  x0 = odd ? r01 : x0; x1 = odd ? x1 : r01;
  x2 = odd ? r23 : x2; x3 = odd ? x3 : r23;
  const float r02 = dpp(hi ? x0 : x2, std::integral_constant<int, 0x4E>{}), r13 = dpp(hi ? x1 : x3, std::integral_constant<int, 0x4E>{});
  x0 = hi ? r02 : x0; x2 = hi ? x2 : r02;
  x1 = hi ? r13 : x1; x3 = hi ? x3 : r13;
#endif
}
template <int J>
__device__ __forceinline__ unsigned quad_broadcast(unsigned v)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mov_dpp(v, J * 0x55, 0xf, 0xf, true);
#else
  return v;
#endif
}
// out: the tensor; at: the lane's image and channel block, in elements.  Called by all lanes of the wave.
template <int A>
__device__ __forceinline__ void store_f32(const float (*y)[(A - 2) * (A - 2)], float *out, size_t at, int g, bool ok, int th, int tw,
                                          int oh_n, int ow_n, int px)
{
  constexpr int M = A - 2;
  typedef float v4f __attribute__((ext_vector_type(4)));
  if constexpr (A == 6) {
    // Four lanes of a quad hold neighbouring tiles: they trade columns, so that an instruction writes the four pixels of a
    // tile's row by sixteen neighbouring lanes -- 256 bytes in one piece, where a lane's own pixel by pixel leaves 64.
    const int lane = threadIdx.x & 63, c = lane & 3;
    const unsigned long long row0 = at + ((unsigned long long)(M * th) * ow_n + M * tw) * px;   // the lane's tile, first pixel
    const int rows = ok ? oh_n - M * th : 0, cols = ow_n - M * tw;                              // pixels of it inside the image
    auto tile = [&](auto jc, const v4f (&v)[4]) {
      constexpr int J = decltype(jc)::value;
      const unsigned long long r = (unsigned long long)quad_broadcast<J>((unsigned)(row0 >> 32)) << 32 | quad_broadcast<J>((unsigned)row0);
      const int nr = (int)quad_broadcast<J>((unsigned)rows), nc = (int)quad_broadcast<J>((unsigned)cols);
      float *p = out + r + (unsigned)(c * px + 4 * g);
      if (c < nc)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          // (non-temporal: output that nothing reads back soon)
          if (i < nr) __builtin_nontemporal_store(v[i], reinterpret_cast<v4f *>(p + (size_t)i * ow_n * px));
    };
    v4f v[4][4];   // [tile of the quad][row]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float x0 = y[k][4 * i], x1 = y[k][4 * i + 1], x2 = y[k][4 * i + 2], x3 = y[k][4 * i + 3];
        quad_transpose4(x0, x1, x2, x3, lane);
        v[0][i][k] = x0; v[1][i][k] = x1; v[2][i][k] = x2; v[3][i][k] = x3;
      }
    tile(std::integral_constant<int, 0>{}, v[0]);
    tile(std::integral_constant<int, 1>{}, v[1]);
    tile(std::integral_constant<int, 2>{}, v[2]);
    tile(std::integral_constant<int, 3>{}, v[3]);
    return;
  }
  if (!ok) return;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const int oh = M * th + i;
    if (oh >= oh_n) break;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int ow = M * tw + j;
      if (ow >= ow_n) break;
      const int e = M * i + j;
      const v4f vv = {y[0][e], y[1][e], y[2][e], y[3][e]};
      __builtin_nontemporal_store(vv, reinterpret_cast<v4f *>(out + at + ((size_t)oh * ow_n + ow) * px + 4 * g));
    }
  }
}

// the one-dimensional output transform of tile sizes 6 and 5
template <int A>
__device__ __forceinline__ void out_1d(const float *f, float *o)
{
  if (A == 6) wino::out6_1d(f, o);
  else wino::out5_1d(f, o);
}

}  // namespace

}  // namespace ehip
#endif
