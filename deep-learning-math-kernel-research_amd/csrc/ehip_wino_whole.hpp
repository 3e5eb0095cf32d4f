// A Winograd layer whole in one kernel: input transform, GEMMs and output transform, with the transformed input of a block of
// tiles in LDS instead of between two kernels.
//
// Replaces, for the layers it takes, the three stages that the reference's fused schedule runs per thread (a161,
// src/elx_int8_conv_wino_xopt.hpp:21-179: elx_conv_wino_trans_input.cpp:599-654, elx_int8_conv_wino_gemm.cpp:23-205,
// elx_conv_wino_trans_output.cpp:212-423); like it, a workgroup takes sixteen tiles through all output channels.
//
// What bounds it: the issue of vector instructions, 1250 per 16 tiles x 16 input channels and 1300 per 16 tiles x 16 output
// channels, the same as the two kernels it replaces; what it saves is what surrounds them, a launch, the start of a kernel
// with cold caches and the way of the transformed input through memory (which is still written, because callers may ask
// the handle for it, but nobody waits for that).  128 -> 128 at 28 x 28, N = 64 (196 blocks, one per CU): 26.7 -> 18.2 us, between other
// layers 24.1 -> 21.5.  Sixteen tiles, not more: a block's tiles at every position fit the LDS up to 256 input
// channels, and at 64 and 128 two or three workgroups do, whose phases then overlap.
// Tried: the tasks of both phases in one list that twelve waves of a persistent workgroup draw from, with up to four
// buffers of tiles and counters in the place of the barrier: 64 -> 64 at 224 x 224 82 us against 79 here, 128 -> 128 at 28 x 28 22 against
// 18; all positions as straight-line code (the wave's 43 KB of instructions miss the instruction cache: 25.0 against 18.4 us).
//
// Compiled with the accumulators in the ordinary vector registers, like ehip_wino_lanes.hip.
#ifndef EHIP_WINO_WHOLE_HPP
#define EHIP_WINO_WHOLE_HPP
#include "ehip_wino_fold.hpp"
#include "ehip_wino_pack.hpp"
#include <type_traits>

namespace ehip {

namespace {

// u8 / s8 output without and with the in-place sum, f32 output
enum { kWholeQuantized, kWholeSum, kWholeF32 };

// bytes of LDS: the transformed tiles [position][4 NKS units][16 tiles][16], and per wave the constants of one group of positions
// (a column of M; tile size 4: all of them) [positions][scale, shift, compensation][4 quads]
constexpr int whole_tile_bytes(int A, int nks) { return A * A * nks * 1024; }
constexpr int whole_const_bytes(int A) { return (A == 4 ? 16 : A) * 12 * 16; }
// waves per SIMD that the registers are shared out for
constexpr int whole_occupancy(int A, int mode, int nks, int nw)
{
  return nw == 4 && mode == kWholeQuantized && 3 * (whole_tile_bytes(A, nks) + 4 * whole_const_bytes(A)) <= 160 * 1024 ? 3 : 2;
}

}  // namespace

// A workgroup takes one block of 16 tiles (and a share of the output channels): its waves transform the units of 16 input
// channels into LDS, meet, and take groups of 16 output channels through all positions.
// a.nx = blocks of 16 tiles, a.splits = workgroups that share a block's output channels, a.per_split = groups of 16 channels of
// each; NKS = k-steps of 64 input channels per position; NW = 8 waves, or 4 where two or three workgroups fit on a CU.
template <int A, int MODE, int NKS, int NW>
__global__ __launch_bounds__(64 * NW, whole_occupancy(A, MODE, NKS, NW)) void k_wino_whole(const WinoWholeArgs *rest, const void *in, void *out, const float *bias_)
{
  constexpr int AA = A * A, M = A - 2, U = 4 * NKS;
  constexpr bool SUM = MODE == kWholeSum;
  WinoArgs wa = load_args(&rest->w);
  WinoFusedArgs a = load_args(&rest->f);
  wa.in = in;
  a.out = out; a.bias = bias_;
  const EHIP_CONSTANT WinoWholeArgs *wc = (const EHIP_CONSTANT WinoWholeArgs *)rest;
  const int nx = wc->nx, splits = wc->splits, per_split = wc->per_split;
  const unsigned nt_magic = wc->nt_magic, wt_magic = wc->wt_magic;
  extern __shared__ float4 lds[];
  constexpr int kTileCells = whole_tile_bytes(A, NKS) / 16, kConstCells = whole_const_bytes(A) / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // neighbouring blocks share input rows and the workgroups of a block its pixels: an XCD takes a run of them
  const int item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (item >= nx * splits) return;   // whole workgroup
  const int blk = item / splits, sp = item - blk * splits;
  const int g_lo = sp * per_split;
  const int g_hi = g_lo + per_split < a.oc2 ? g_lo + per_split : a.oc2;
  const int l16 = lane & 15, g = lane >> 4, q = lane & 3, tl = lane >> 2;

  // ---- input transform: a wave takes units of 16 channels, a lane one tile x four channels ----------------------
  {
    int t = blk * 16 + tl;
    t = t < a.t ? t : a.t - 1;         // (a lane without a tile takes part with the last one)
    TileCoord c;
    c.n = fastdiv_any(t, a.nt, nt_magic);
    const int rem = t - c.n * a.nt;
    c.th = fastdiv_any(rem, a.wt, wt_magic);
    c.tw = rem - c.th * a.wt;
    c.h0 = M * c.th - wa.pad_t;
    c.w0 = M * c.tw - wa.pad_l;
    c.border = c.h0 < 0 || c.w0 < 0 || c.h0 + A - 1 >= wa.ih || c.w0 + A - 1 >= wa.iw;
    // (the pixels of a unit pass through the place of its transformed tiles)
    if constexpr (2 * U <= NW) {
      // twice as many waves as units: two waves share a unit's pixels and take two channels of every quad each
      const int u = wave >> 1;
      uint4 *cells = reinterpret_cast<uint4 *>(lds) + u * 16;
      unsigned *quads = reinterpret_cast<unsigned *>(cells + tl) + q;
      unsigned packed[AA];
      if (u < a.ic2) gather_tile_lds<A, 16 * U, 2>(wa, c, u, q, tl, cells, wave & 1);
      __syncthreads();                   // the pixels are in LDS
      if (u < a.ic2) quantize_tile_lds<A, 16 * U, 2>(quads, c.border, wa.mrepS, wa.mz, packed, 2 * (wave & 1));
      __syncthreads();                   // and read
      unsigned short *pairs = reinterpret_cast<unsigned short *>(quads) + (wave & 1);
      if (u < a.ic2)
#pragma unroll
        for (int e = 0; e < AA; ++e) pairs[128 * U * e] = (unsigned short)(packed[e] ^ 0x8080u);
    } else {
      for (int u = wave; u < a.ic2; u += NW) {
        uint4 *cells = reinterpret_cast<uint4 *>(lds) + u * 16;
        unsigned *quads = reinterpret_cast<unsigned *>(cells + tl) + q;
        unsigned packed[AA];
        gather_tile_lds<A, 16 * U>(wa, c, u, q, tl, cells);
        quantize_tile_lds<A, 16 * U>(quads, c.border, wa.mrepS, wa.mz, packed);
#pragma unroll
        for (int e = 0; e < AA; ++e) quads[64 * U * e] = packed[e] ^ 0x80808080u;
      }
    }
  }

  // ---- GEMMs and output transform: a wave takes groups of 16 output channels -------------------------------------
  // A group of positions (a column of M, rows inside, both in Fold's order; tile size 4: all positions in order) is
  // straight-line code, the groups are a loop: the instructions of all positions would not stay in the instruction cache.
  constexpr int NCOL = A == 4 ? 1 : A, PER = AA / NCOL, SC = PER * NKS;   // groups, positions and steps of a group
  constexpr int D = A == 6 ? 6 : (A == 5 ? 5 : 8);                        // ring of weights; divides SC
  static_assert(SC % D == 0, "ring");
  constexpr int CELLS = PER * 12, NC = (CELLS + 63) / 64;
  auto row_order = [](int i) { return A == 4 ? i : (int)Fold<A>::kOrder[i % A]; };
  // the group's 16 channels are one block of the output: of the group of 32 packed rows (row 8 gq + 4 h + j holds channel
  // 16 h + 4 gq + j) it takes the rows of half h
  // (the launcher checks that the packed weights are addressed with 32 bits)
  const unsigned a_row = (unsigned)(g * a.ocpp + 8 * (l16 >> 2) + (l16 & 3)) * 16u;
  const unsigned w_ks = (unsigned)a.ocpp * 64u, w_pos = (unsigned)a.units_pad * (unsigned)a.ocpp * 16u;
  const BufferRsrc rw = make_rsrc(a.w, AA * w_pos);
  auto weights_of = [&](int gi, int ci) {   // of the ci-th column of channel block gi
    return (unsigned)((gi >> 1) * 512 + (gi & 1) * 64) + (A == 4 ? 0u : (unsigned)Fold<A>::order(ci)) * w_pos;
  };
  v4i ra[D];
  auto issue = [&](int sn, unsigned wb, unsigned pos) {   // step sn of a column; pos: w_pos
    buffer_load_cell(rw, a_row, wb + (unsigned)(A == 4 ? sn / NKS : A * row_order(sn / NKS)) * pos + (unsigned)(sn % NKS) * w_ks, ra[sn % D]);
  };
  // constants: cell = (position of the column, array, quad), lane + 64 j of them for a lane; its offset in the first column of
  // memory.  (A lane without a j-th cell takes the last one again, and stores nothing.)
  auto c_off = [&](int j) {
    int idx = lane + 64 * j;
    idx = idx < CELLS ? idx : CELLS - 1;
    const int r = idx / 12, rem = idx - 12 * r, arr = rem >> 2, gq = rem & 3;
    return (arr * AA + (A == 4 ? r : A * r)) * a.ocpp + 4 * gq;
  };
  const int c_off0 = c_off(0), c_off1 = c_off(1), c_off2 = c_off(2);
  float4 cst0, cst1, cst2;
  auto request_consts = [&](int gi, int ci) {
    const float *src = a.scale + (long long)(A == 4 ? 0 : Fold<A>::order(ci)) * a.ocpp + gi * 16;
    cst0 = *reinterpret_cast<const float4 *>(src + c_off0);
    if constexpr (NC > 1) cst1 = *reinterpret_cast<const float4 *>(src + c_off1);
    if constexpr (NC > 2) cst2 = *reinterpret_cast<const float4 *>(src + c_off2);
  };
  const int cl0 = kTileCells + wave * kConstCells;   // the wave's constants, in cells
  auto store_consts = [&]() {
    if (CELLS >= 64 || lane < CELLS) lds[cl0 + lane] = cst0;
    if constexpr (NC > 1)
      if (CELLS >= 128 || lane + 64 < CELLS) lds[cl0 + lane + 64] = cst1;
    if constexpr (NC > 2)
      if (CELLS >= 192 || lane + 128 < CELLS) lds[cl0 + lane + 128] = cst2;
  };
  int gi = g_lo + wave;
  unsigned wb = weights_of(gi < g_hi ? gi : g_lo, 0);
  if (gi < g_hi) {
    request_consts(gi, 0);
#pragma unroll
    for (int k = 0; k < D; ++k) issue(k, wb, w_pos);
  }
  // the transformed tiles are in LDS (nothing waits for the loads above)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");

  const int t = blk * 16 + l16;
  const int tc = t < a.t ? t : 0;
  const int n = fastdiv_any(tc, a.nt, nt_magic);
  const int rem = tc - n * a.nt;
  const int th = fastdiv_any(rem, a.wt, wt_magic);
  const int tw = rem - th * a.wt;
  const bool valid = t < a.t;
  const int px = a.out_nhwc ? a.oc2 * 16 : 16;
  int clg = cl0 + g;   // cells; opaque, so that reads are base + immediate offset
  asm volatile("" : "+v"(clg));
  const v4i *vl = reinterpret_cast<const v4i *>(lds);
  for (; gi < g_hi; gi += NW) {
    const bool more = gi + NW < g_hi;                      // wave-uniform
    float Y[4][M][4];                // [channel][row][running values of the second dimension]
    float C[4][4];                   // [channel][running values of the first dimension]
    float P[A == 4 ? AA : 1][4];     // tile size 4: the requantized positions
    if constexpr (A != 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
          for (int j = 0; j < 4; ++j) asm volatile("" : "=v"(Y[k][r][j]));   // (written before it is read, in the loop's first rounds)
    }
    auto column = [&](int ci) {
      store_consts();
      const bool last = ci == NCOL - 1;
      const int gn = last && more ? gi + NW : gi, cn = last ? 0 : ci + 1;
      const unsigned wbn = weights_of(gn, cn);   // (behind the last column: its group's head again, unused)
      unsigned pos = w_pos;
      asm volatile("" : "+s"(pos));   // (the steps' offsets are worked out where they are used, not kept for all columns)
      const int v0 = lane + (A == 4 ? 0 : Fold<A>::order(ci)) * (U * 16);
      auto vcell = [&](int sn) { return (A == 4 ? sn / NKS : A * row_order(sn / NKS)) * (U * 16) + sn % NKS * 64; };
      v4i acc[2], rb[3];
      float4 sc[2], sh[2];
      rb[0] = vl[v0 + vcell(0)];
      if (SC > 1) rb[1] = vl[v0 + vcell(1)];
      request_consts(gn, cn);
      auto finish = [&](int ri) {
        const float scv[4] = {sc[ri & 1].x, sc[ri & 1].y, sc[ri & 1].z, sc[ri & 1].w};
        const float shv[4] = {sh[ri & 1].x, sh[ri & 1].y, sh[ri & 1].z, sh[ri & 1].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float x = __builtin_fmaf((float)acc[ri & 1][k], scv[k], shv[k]);
          if constexpr (A == 4) {
            P[ri][k] = x;
            asm volatile("" : "+v"(P[ri][k]));
          } else {
            fold_step<A>(ri, C[k], x, std::make_integer_sequence<int, A>{});
            pin(C[k], ri);   // (left to itself the compiler defers the folding and keeps every requantized value instead)
          }
        }
      };
#pragma unroll
      for (int ri = 0; ri < PER; ++ri) {
        const int cr = clg + 12 * (A == 4 ? ri : row_order(ri));
        // (the accumulators start from the compensation 128 * sum(weights) of their (position, channel))
        const float4 cf = lds[cr + 8];
        acc[ri & 1] = v4i{__float_as_int(cf.x), __float_as_int(cf.y), __float_as_int(cf.z), __float_as_int(cf.w)};
        sc[ri & 1] = lds[cr];
        sh[ri & 1] = lds[cr + 4];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const int sn = ri * NKS + ks;
          if (sn + 2 < SC) rb[(sn + 2) % 3] = vl[v0 + vcell(sn + 2)];   // the tiles of the step after next
          acc[ri & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ra[sn % D], rb[sn % 3], acc[ri & 1], 0, 0, 0);
          if (sn + D < SC) issue(sn + D, wb, pos);
          else issue(sn + D - SC, wbn, pos);
          if (ks == 0 && ri > 0) finish(ri - 1);   // (between the matrix instructions of the next position)
          __builtin_amdgcn_sched_barrier(0);       // (the loads stay where the ring puts them)
        }
      }
      finish(PER - 1);
      wb = wbn;
    };
    if constexpr (A == 4) column(0);
    else {
#pragma unroll 1
      for (int ci = 0; ci < A; ++ci) {
        column(ci);
        // the second fold differs from column to column: separate blocks, each with an opaque statement inside, or they
        // become selects between all of them
        auto fold_rows = [&](auto kc_) {
          constexpr int K = decltype(kc_)::value;
          int c = ci;
          asm volatile("" : "+s"(c));   // (every test stands alone)
          if (c == K) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
              for (int r = 0; r < M; ++r) Fold<A>::template step_in_place<K>(Y[k][r], Fold<A>::result(C[k], r));
          }
        };
        fold_rows(std::integral_constant<int, 0>{});
        fold_rows(std::integral_constant<int, 1>{});
        fold_rows(std::integral_constant<int, 2>{});
        fold_rows(std::integral_constant<int, 3>{});
        fold_rows(std::integral_constant<int, 4>{});
        if (A == 6) fold_rows(std::integral_constant<int, A - 1>{});
      }
    }
    // ---- output: bias, output scale, old output, ReLU, rounding; whole cells --------------------------------
    float4 bias = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.with_bias) bias = *reinterpret_cast<const float4 *>(a.bias + 16 * gi + 4 * g);
    const size_t plane = a.out_nhwc ? (size_t)n * a.oh * a.ow * a.oc2 * 16 + gi * 16 : ((size_t)n * a.oc2 + gi) * a.oh * a.ow * 16;
    auto value = [&](int k, float *y) {
      if constexpr (A == 4) {
        float f[AA];
#pragma unroll
        for (int q = 0; q < AA; ++q) f[q] = P[q][k];
        wino::tile_output<4>(f, y);
      } else {
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
          for (int c = 0; c < M; ++c) y[M * r + c] = Fold<A>::result(Y[k][r], c);
      }
    };
    if constexpr (MODE == kWholeF32) {
      float y[4][M * M];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        value(k, y[k]);
        finish_channel_f32<A>(y[k], comp_of(bias, k), a.with_bias != 0, a.with_relu != 0);
#pragma unroll
        for (int q = 0; q < M * M; ++q) asm volatile("" : "+v"(y[k][q]));
        __builtin_amdgcn_sched_barrier(0);
      }
      store_f32<A>(y, static_cast<float *>(a.out), plane, g, valid, th, tw, a.oh, a.ow, px);
    } else {
      uint8_t *block = static_cast<uint8_t *>(a.out) + plane;
      unsigned pk[M * M], old[M * M];
#pragma unroll
      for (int q = 0; q < M * M; ++q) pk[q] = 0u;
      if (SUM) load_old_cells<A>(old, block, g, th, tw, a.oh, a.ow, px);
      auto quantize = [&](auto out_c, auto relu_c) {
        constexpr int OUT = decltype(out_c)::value;
        constexpr bool RELU = decltype(relu_c)::value;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float y[M * M];
          value(k, y);
          pack_channel<OUT, A>(y, comp_of(bias, k), k, RELU, a.out_repS, a.out_z, SUM, old, pk);
#pragma unroll
          for (int q = 0; q < M * M; ++q) asm volatile("" : "+v"(pk[q]));
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      using U8C = std::integral_constant<int, EHIP_U8>;
      using S8C = std::integral_constant<int, EHIP_S8>;
      if (a.out_type == EHIP_U8) {
        if (a.with_relu) quantize(U8C{}, std::true_type{});
        else quantize(U8C{}, std::false_type{});
      } else {
        if (a.with_relu) quantize(S8C{}, std::true_type{});
        else quantize(S8C{}, std::false_type{});
      }
      store_cells<A>(pk, block, g, valid, th, tw, a.oh, a.ow, px);
    }
  }
  // the handle's transformed input, as the stand-alone transform leaves it: [t / 32][position][unit][32][16].  Last of all, since a
  // wave's loads and stores are waited for in order: ahead of the GEMMs their weights waited for these stores, too (128 -> 128 at
  // 28 x 28 between other layers 23.5 us that way, 21.5 this).
  if (sp == 0) {
    uint8_t *tin = const_cast<uint8_t *>(a.tin) + (long long)(blk >> 1) * AA * a.ic2 * 512 + ((blk & 1) * 16 + l16) * 16;
    for (int p = wave; p < AA; p += NW)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (4 * ks + g < a.ic2) {
          typedef float v4f __attribute__((ext_vector_type(4)));
          const float4 v = lds[(p * U + 4 * ks) * 16 + lane];
          __builtin_nontemporal_store(v4f{v.x, v.y, v.z, v.w}, reinterpret_cast<v4f *>(tin + ((long long)p * a.ic2 + 4 * ks + g) * 512));
        }
  }
}

template <int A>
WholeForm whole_form(int nks, int nw, int out_type, bool sum)
{
#define EHIP_WHOLE(NKS, NW)                                                                                              \
  WholeForm{out_type == EHIP_F32 ? k_wino_whole<A, kWholeF32, NKS, NW>                                                   \
                                 : sum ? k_wino_whole<A, kWholeSum, NKS, NW> : k_wino_whole<A, kWholeQuantized, NKS, NW>, \
            NW, whole_tile_bytes(A, NKS) + NW * whole_const_bytes(A)}
  switch (nks) {
    case 1: return nw == 4 ? EHIP_WHOLE(1, 4) : EHIP_WHOLE(1, 8);
    case 2: return nw == 4 ? EHIP_WHOLE(2, 4) : EHIP_WHOLE(2, 8);
    case 3: return EHIP_WHOLE(3, 8);
    default: return EHIP_WHOLE(4, 8);
  }
#undef EHIP_WHOLE
}

}  // namespace ehip
#endif
