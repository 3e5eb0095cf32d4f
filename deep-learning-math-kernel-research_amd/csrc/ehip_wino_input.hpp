// The input side of a Winograd layer: a tile's pixels from the user's tensor, V = Bt d B, and the u8 codes of the
// transformed tile.  Shared by the stand-alone input transform (ehip_wino.hip) and by the kernel that runs a layer whole
// (ehip_wino_whole.hpp); a lane holds one tile x four channels.
#ifndef EHIP_WINO_INPUT_HPP
#define EHIP_WINO_INPUT_HPP
#include "ehip_internal.hpp"
#include "ehip_wino_tiles.hpp"
#include <type_traits>

namespace ehip {

namespace {

// Buffer addressing (a load whose offset lies outside the buffer returns zero and touches no memory).  The
// builtins exist in the device pass only.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
__device__ __forceinline__ BufferRsrc make_rsrc(const void *base, unsigned bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void buffer_load_cell(BufferRsrc r, unsigned off, float4 &v)
{
  typedef float v4f __attribute__((ext_vector_type(4)));
  const v4f x = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  v = make_float4(x.x, x.y, x.z, x.w);
}
__device__ __forceinline__ void buffer_load_cell(BufferRsrc r, unsigned off, unsigned &v)
{
  v = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}
__device__ __forceinline__ void buffer_load_cell(BufferRsrc r, unsigned off, uint4 &v)
{
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  const v4u x = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  v = make_uint4(x.x, x.y, x.z, x.w);
}
__device__ __forceinline__ void buffer_load_cell(BufferRsrc r, unsigned off, float2 &v)
{
  typedef float v2f __attribute__((ext_vector_type(2)));
  const v2f x = __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
  v = make_float2(x.x, x.y);
}
// (off: the lane's bytes, checked against the buffer; at: a wave-uniform offset on top)
__device__ __forceinline__ void buffer_load_cell(BufferRsrc r, unsigned off, unsigned at, v4i &v)
{
  v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)at, 0));
}
#else
typedef int BufferRsrc;
__device__ inline BufferRsrc make_rsrc(const void *, unsigned) { return 0; }
__device__ inline void buffer_load_cell(BufferRsrc, unsigned, float4 &v) { v = float4(); }
__device__ inline void buffer_load_cell(BufferRsrc, unsigned, float2 &v) { v = float2(); }
__device__ inline void buffer_load_cell(BufferRsrc, unsigned, unsigned &v) { v = 0u; }
__device__ inline void buffer_load_cell(BufferRsrc, unsigned, uint4 &v) { v = uint4(); }
__device__ inline void buffer_load_cell(BufferRsrc, unsigned, unsigned, v4i &v) { v = v4i(); }
#endif

__device__ __forceinline__ float comp_of(const float4 &v, int k)
{
  return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w));
}

__device__ __forceinline__ float comp_of(const float2 &v, int k) { return k == 0 ? v.x : v.y; }

// four u8 codes in a dword: the reference turns the codes into floats as they are
// (src/kernel/elk_conv_wino_4x4_3x3_input.hxx:40-47)
__device__ __forceinline__ float comp_of(const unsigned &v, int k)
{
  return (float)((v >> (8 * k)) & 0xffu);
}

struct TileCoord {
  int n, th, tw, h0, w0;
  bool border;
};
template <int A>
__device__ __forceinline__ TileCoord tile_coord(const WinoArgs &a, int t)
{
  TileCoord c;
  c.n = t / a.nt;
  const int rem = t - c.n * a.nt;
  c.th = rem / a.wt;
  c.tw = rem - c.th * a.wt;
  c.h0 = (A - 2) * c.th - a.pad_t;
  c.w0 = (A - 2) * c.tw - a.pad_l;
  c.border = c.h0 < 0 || c.w0 < 0 || c.h0 + A - 1 >= a.ih || c.w0 + A - 1 >= a.iw;
  return c;
}

// the lane's four channels of the A x A pixels of a tile: float4 (f32 input) or 4 packed codes (u8)
template <int A>
__device__ __forceinline__ void gather_tile(const WinoArgs &a, const TileCoord &c, int c2, int q, float4 *d)
{
  // blocked: the 16-channel plane of (n, c2), 4 quads per pixel; nhwc: quad c2 * 4 + q of every pixel's vector
  const size_t pq = a.in_nhwc ? (size_t)a.ic2 * 4 : 4;   // quads between neighbouring pixels
  const float4 *plane = reinterpret_cast<const float4 *>(a.in) +
      (a.in_nhwc ? (size_t)c.n * a.ih * a.iw * pq + c2 * 4 : ((size_t)c.n * a.ic2 + c2) * a.ih * a.iw * 4) + q;
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < A; ++j) {
      const int h = c.h0 + i, w = c.w0 + j;
      d[A * i + j] = (h >= 0 && h < a.ih && w >= 0 && w < a.iw) ? plane[((size_t)h * a.iw + w) * pq]
                                                                   : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
template <int A>
__device__ __forceinline__ void gather_tile(const WinoArgs &a, const TileCoord &c, int c2, int q, unsigned *d)
{
  const size_t pq = a.in_nhwc ? (size_t)a.ic2 * 4 : 4;
  const unsigned *plane = reinterpret_cast<const unsigned *>(a.in) +
      (a.in_nhwc ? (size_t)c.n * a.ih * a.iw * pq + c2 * 4 : ((size_t)c.n * a.ic2 + c2) * a.ih * a.iw * 4) + q;
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < A; ++j) {
      const int h = c.h0 + i, w = c.w0 + j;
      d[A * i + j] = (h >= 0 && h < a.ih && w >= 0 && w < a.iw) ? plane[((size_t)h * a.iw + w) * pq] : 0u;   // the frame is 0.0f
    }
}

// The same gather through buffer addressing, for tensors below 4 GB (WinoArgs::buf_gather).  A cell's byte
// offset is the lane's first cell's (32 bits, possibly "negative" for a tile that starts in the frame) plus
// a scalar; rows and columns are tested once each, a cell's test is the AND of two lane masks (scalar
// instructions), and a cell of the frame is sent to an offset outside the buffer, where the load returns
// the frame's zero.  Two vector instructions per cell instead of a bounds test, a 64-bit multiply-add and
// a branch.
template <int A, typename Cell>
__device__ __forceinline__ void gather_tile_buf(const WinoArgs &a, const TileCoord &c, int c2, int q, Cell *d)
{
  const unsigned pq = a.in_nhwc ? (unsigned)a.ic2 * 4u : 4u;   // cells between neighbouring pixels
  const unsigned cells = (unsigned)a.n * a.ic2 * a.ih * a.iw * 4u;
  const BufferRsrc rin = make_rsrc(a.in, cells * (unsigned)sizeof(Cell));
  const unsigned plane = a.in_nhwc ? (unsigned)c.n * a.ih * a.iw * pq + c2 * 4u
                                   : ((unsigned)c.n * a.ic2 + c2) * a.ih * a.iw * 4u;
  const unsigned voff = (plane + (unsigned)(c.h0 * a.iw + c.w0) * pq + q) * (unsigned)sizeof(Cell);
  bool rv[A], cv[A];
#pragma unroll
  for (int i = 0; i < A; ++i) {
    rv[i] = (unsigned)(c.h0 + i) < (unsigned)a.ih;
    cv[i] = (unsigned)(c.w0 + i) < (unsigned)a.iw;
  }
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < A; ++j) {
      const unsigned so = (unsigned)(i * a.iw + j) * pq * (unsigned)sizeof(Cell);   // scalar
      buffer_load_cell(rin, (rv[i] && cv[j]) ? voff + so : 0xffffff00u, d[A * i + j]);
    }
}
// The lane's two channels (o2: their place among a unit's eight pairs) of an f32 tensor of at most 2^30 - 2^24 bytes.  A row and a column
// outside the image each add enough to leave the buffer, and their sum does not come round, so that an address is one addition.
template <int A>
__device__ __forceinline__ void gather_tile_pairs(const WinoArgs &a, const TileCoord &c, int c2, int o2, float2 *d)
{
  const unsigned px = a.in_nhwc ? (unsigned)a.ic2 * 64u : 64u;   // bytes between neighbouring pixels
  const BufferRsrc rin = make_rsrc(a.in, (unsigned)a.n * a.ic2 * a.ih * a.iw * 64u);
  const unsigned plane = a.in_nhwc ? (unsigned)c.n * a.ih * a.iw * px + c2 * 64u : ((unsigned)c.n * a.ic2 + c2) * a.ih * a.iw * 64u;
  const unsigned at = plane + (unsigned)(c.h0 * a.iw + c.w0) * px + (unsigned)o2 * 8u, row = (unsigned)a.iw * px;
  unsigned ro[A], co[A];
#pragma unroll
  for (int i = 0; i < A; ++i) {
    ro[i] = (unsigned)(c.h0 + i) < (unsigned)a.ih ? at + i * row : 0x80000000u;
    co[i] = (unsigned)(c.w0 + i) < (unsigned)a.iw ? i * px : 0x40000000u;
  }
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < A; ++j) buffer_load_cell(rin, ro[i] + co[j], d[A * i + j]);
}


// u8 input below 4 GB, by whole cells and through LDS: `cells` = the wave's own [A x A pixels][16 tiles] cells of 16 bytes, S
// cells from pixel to pixel.  Lane (tile, q) fetches the cells (all four channel quads) of pixels q, 4 + q, ... of its tile --
// a wave's load covers 16 tiles x four neighbouring pixels, a quarter of the load instructions and of the cache lines looked
// up per byte that a dword per lane and pixel costs -- and later reads back its own quad of every pixel: LDS reads with
// immediate offsets in the place of the 144 vector instructions of a 4 x 4 exchange inside the quad.  Only the wave's own
// lanes meet in `cells`, and a wave's LDS operations are done in order: no barrier.  Cells of the zero frame are sent to an
// offset outside the buffer, as in gather_tile_buf.  (P waves that share the cells: a wave makes every P-th load, from the k0-th on,
// and they meet at a barrier.)
template <int A, int S = 16, int P = 1>
__device__ __forceinline__ void gather_tile_lds(const WinoArgs &a, const TileCoord &c, int c2, int q, int tl, uint4 *cells, int k0 = 0)
{
  constexpr int AA = A * A, NK = ((AA + 3) / 4 + P - 1) / P;
  const unsigned pc = a.in_nhwc ? (unsigned)a.ic2 : 1u;   // cells between neighbouring pixels
  const BufferRsrc rin = make_rsrc(a.in, (unsigned)a.n * a.ic2 * a.ih * a.iw * 16u);
  const unsigned plane = a.in_nhwc ? (unsigned)c.n * a.ih * a.iw * pc + c2 : ((unsigned)c.n * a.ic2 + c2) * a.ih * a.iw;
  uint4 v[NK];
  int e0 = 4 * k0 + q;               // the lane's first pixel, 4 P further on the next
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int e = e0 + 4 * P * k;
    const int i = e / A, j = e - A * i;
    const int h = c.h0 + i, w = c.w0 + j;
    const bool ok = e < AA && (unsigned)h < (unsigned)a.ih && (unsigned)w < (unsigned)a.iw;
    const unsigned off = (plane + (unsigned)(h * a.iw + w) * pc) * 16u;
    buffer_load_cell(rin, ok ? off : 0xffffff00u, v[k]);
  }
  uint4 *mine = cells + e0 * S + tl;
#pragma unroll
  for (int k = 0; k < NK; ++k)
    if (4 * P * (k + 1) <= AA || e0 + 4 * P * k < AA) mine[4 * P * S * k] = v[k];
  __builtin_amdgcn_wave_barrier();
}

// min(s, a, b) in one instruction (left to itself the compiler pairs the values up first: three for four values, not two)
__device__ __forceinline__ float min3(float s, float a, float b)
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_min3_f32 %0, %0, %1, %2" : "+v"(s) : "v"(a), "v"(b));
#endif
  return s;
}
// the same with a NaN for a NaN
__device__ __forceinline__ float minimum3(float s, float a, float b)
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_minimum3_f32 %0, %0, %1, %2" : "+v"(s) : "v"(a), "v"(b));
#endif
  return s;
}
// packed[position]: the lane's four (float2 cells: two) channels of the transformed tile as u8 codes.
template <typename Cell, int A>
__device__ __forceinline__ void quantize_tile(const Cell *d, bool border, float mrepS, float mz, unsigned *packed)
{
  constexpr int AA = A * A;
  constexpr bool kCodes = sizeof(Cell) == sizeof(unsigned);
  constexpr int kChannels = sizeof(Cell) == sizeof(float2) ? 2 : 4;
  // mixed: the wave holds interior and rim tiles -- the per-lane, branch-free form of the transform.
  // Quantization: sat_u8(rne_to_u32(V * (in_S / tin_S) + tin_z)), one rounding in the multiply-add.  The
  // reference's float -> u32 conversion turns everything below -0.5 (and NaN) into 0xffffffff, which then
  // saturates to 255; v_cvt_pk_u8_f32 rounds to nearest even and saturates the rest.  watch: the plain
  // conversion, with the quirk's cases only looked for: a running minimum that a NaN sticks to, an instruction per two values,
  // says whether one was seen (never, with a calibrated tinput_quant); the caller then runs the exact form again.
  // u8 user input: the codes are finite, so with finite quantization constants no NaN can arise; constants that are not
  // finite send every wave to the exact form.
  const bool odd_consts = !(__builtin_fabsf(mrepS) <= 3.402823466e38f) || !(__builtin_fabsf(mz) <= 3.402823466e38f);
  auto channels = [&](bool mixed, bool watch) {
    float seen = 0.0f;
#pragma unroll
    for (int k = 0; k < AA; ++k) packed[k] = 0u;
#pragma unroll
    for (int k = 0; k < kChannels; ++k) {
      float f[AA], v[AA];
#pragma unroll
      for (int e = 0; e < AA; ++e) f[e] = comp_of(d[e], k);
      if (kCodes || mixed) wino::tile_input_lanes<A, kCodes>(f, v, border);
      else wino::tile_input<A>(f, v, false);
      if (watch) {
        float y[AA];
#pragma unroll
        for (int e = 0; e < AA; ++e) {
          y[e] = __builtin_fmaf(v[e], mrepS, mz);
          packed[e] = __builtin_amdgcn_cvt_pk_u8_f32(y[e], k, packed[e]);
        }
#pragma unroll
        for (int e = 0; e + 1 < AA; e += 2) seen = kCodes ? __builtin_fminf(seen, __builtin_fminf(y[e], y[e + 1])) : minimum3(seen, y[e], y[e + 1]);
        if (AA & 1) seen = kCodes ? __builtin_fminf(seen, y[AA - 1]) : minimum3(seen, y[AA - 1], y[AA - 1]);
      } else {
#pragma unroll
        for (int e = 0; e < AA; ++e) {
          const float y = __builtin_fmaf(v[e], mrepS, mz);
          packed[e] = __builtin_amdgcn_cvt_pk_u8_f32(y >= -0.5f ? y : 300.0f, k, packed[e]);
        }
      }
    }
    return kCodes ? (seen < -0.5f || odd_consts) : !(seen >= -0.5f);
  };
  const bool mixed = !kCodes && __ballot(border) != 0;   // wave-uniform
  bool again;
  if (mixed) again = channels(true, true);
  else again = channels(false, true);
  if (__ballot(again) != 0) {
    if (mixed) channels(true, false);
    else channels(false, false);
  }
}

// The same for the pixels that gather_tile_lds left in LDS (quads: the lane's, 4 S dwords from pixel to pixel), with few
// registers: every channel reads its bytes, column by column, and a row of the result is packed as it is finished.  At 128
// registers four waves fit on a SIMD.  (CH < 4: that many channels of the quad, from the k0-th on, in the low bytes.)  The channels are a loop: a quarter of the instructions to fetch, which a layer between
// other layers finds in no cache.
template <int A, int S = 16, int CH = 4>
__device__ __forceinline__ void quantize_tile_lds(const unsigned *quads, bool border, float mrepS, float mz, unsigned *packed, int k0 = 0)
{
  constexpr int AA = A * A;
  const bool odd_consts = !(__builtin_fabsf(mrepS) <= 3.402823466e38f) || !(__builtin_fabsf(mz) <= 3.402823466e38f);
  auto channels = [&](auto exact_c) {
    constexpr bool EXACT = decltype(exact_c)::value;
    float seen = 0.0f;
#pragma unroll
    for (int e = 0; e < AA; ++e) packed[e] = 0u;
    const uint8_t *bytes = reinterpret_cast<const uint8_t *>(quads) + k0;
#pragma unroll 1
    for (int k = 0; k < CH; ++k, ++bytes) {
      auto pack = [&](int e, float v) {
        const float y = __builtin_fmaf(v, mrepS, mz);
        packed[e] = __builtin_amdgcn_cvt_pk_u8_f32(!EXACT || y >= -0.5f ? y : 300.0f, k, packed[e]);
        return y;
      };
      if constexpr (A == 4) {
        float f[AA], v[AA], y[AA];
#pragma unroll
        for (int e = 0; e < AA; ++e) f[e] = (float)bytes[16 * S * e];
        wino::tile_input<4>(f, v, border);
#pragma unroll
        for (int e = 0; e < AA; ++e) y[e] = pack(e, v[e]);
#pragma unroll
        for (int e = 0; e < AA; e += 2) seen = min3(seen, y[e], y[e + 1]);
      } else {
        float m[AA];
#pragma unroll
        for (int j = 0; j < A; ++j) {
          float f[A], o[A];
#pragma unroll
          for (int i = 0; i < A; ++i) f[i] = (float)bytes[16 * S * (A * i + j)];
          wino::codes_column<A>(f, o);
#pragma unroll
          for (int i = 0; i < A; ++i) m[A * i + j] = o[i];
        }
#pragma unroll
        for (int i = 0; i < A; ++i) {
          float v[A], y[A];
          wino::codes_row<A>(i, &m[A * i], v, border);
#pragma unroll
          for (int j = 0; j < A; ++j) y[j] = pack(A * i + j, v[j]);
#pragma unroll
          for (int j = 0; j + 1 < A; j += 2) seen = min3(seen, y[j], y[j + 1]);
          if (A & 1) seen = __builtin_fminf(seen, y[A - 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    return seen < -0.5f || odd_consts;
  };
  // (the exact conversion only where a wave saw a value below -0.5: see quantize_tile)
  if (__ballot(channels(std::false_type{})) != 0) channels(std::true_type{});
}

}  // namespace

}  // namespace ehip
#endif
