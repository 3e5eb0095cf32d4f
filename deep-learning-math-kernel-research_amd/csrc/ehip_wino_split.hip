// Winograd GEMMs + output transform for few output values: the input channels of a small block shared out among the waves of a
// workgroup.
//
// Replaces, for those layers, elx_int8_conv_wino_gemm_t::execute + trans_output as the reference's fused schedule
// runs them per thread (a161, src/elx_int8_conv_wino_xopt.hpp:21-179; src/elx_int8_conv_wino_gemm.cpp:23-205,
// src/elx_conv_wino_trans_output.cpp:212-423).
//
// Compiled with the accumulators in the ordinary vector registers, like ehip_wino_lanes.hip.
#include "ehip_wino_pack.hpp"
#include <type_traits>

namespace ehip {

// A layer of few tiles is bound by the chain of one workgroup: the ring kernels take 20 us for a block of 32 channels x 32 tiles
// with 512 input channels, alone on the chip or not, because every k-step of every position passes through the LDS (2 KB of
// reads for a matrix instruction) one after the other, and half of the CUs or more have no block.  Here a workgroup owns 16
// output channels x 16 tiles at all positions, and its wave w the w-th k-step of 64 input channels: one matrix instruction per
// position, whose operands come straight from memory, up to eighteen positions ahead.  The waves' partial sums (integers: exact
// in any order) meet in LDS column by column; there a lane of the first four waves owns one tile x one channel, adds its parts
// up, requantizes, and runs the output transform of that one channel; the finished values go through LDS once more and leave by
// whole cells.  512 -> 512, 256 tiles of 14 x 14 images: 20.4 -> 11.4 us; 256 -> 256 at 28 x 28, N = 1 11.4 -> 7.9.  The price is the
// traffic, 2 KB for a matrix instruction through the L1 and L2 of a CU: a second round of workgroups costs as much as the
// ring kernels' first (512 workgroups 29 us).
// Tried: 32 channels a workgroup, which reads a quarter less: the parts fill the LDS, and adding them up takes twice as long
// (16 against 11 us alone, 21.6 against 21.2 of the ring kernels at 256 workgroups).
// a.nx = blocks of 16 tiles, a.ny = groups of 16 channels; a.slots != 0: an XCD takes every eighth group of channels with all
// tiles, else every eighth block of tiles with all channels (whichever leaves it less to read).
template <int A, int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_wino_gemm_output_lanes_split(const WinoFusedArgs *rest, void *out, const float *bias_)
{
  WinoFusedArgs a = load_args(rest);
  a.out = out; a.bias = bias_;
  constexpr int AA = A * A, M = A - 2, MM = M * M, TB = 64 * NW;
  constexpr int D = A == 4 ? AA : 3 * A;       // positions ahead
  __shared__ v4i part[2][A][NW][64];
  __shared__ float cst[3][AA][16];             // scale, shift, compensation
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int by = a.slots ? seq / a.nx * 8 + xcd : seq % a.ny;
  const int bx = a.slots ? seq % a.nx : seq / a.ny * 8 + xcd;
  if (bx >= a.nx || by >= a.ny) return;        // whole workgroup
  // the workgroup's 16 channels are one block of the output: of the group of 32 packed rows (row 8 gq + 4 h + j holds channel
  // 16 h + 4 gq + j) the rows of half h
  const unsigned w_pos = (unsigned)a.units_pad * (unsigned)a.ocpp * 16u, t_pos = (unsigned)a.ic2 * 512u;   // bytes (the launcher
  const BufferRsrc rw = make_rsrc(a.w, AA * w_pos), rt = make_rsrc(a.tin, (unsigned)((a.t + 31) >> 5) * AA * t_pos);   // checks 32 bits)
  int u = 4 * wave + g;
  const unsigned a_off = (unsigned)(u * a.ocpp + (by >> 1) * 32 + (by & 1) * 4 + 8 * (l16 >> 2) + (l16 & 3)) * 16u;
  u = u < a.ic2 ? u : a.ic2 - 1;               // (units past the last real one multiply zero weights: any cell will do)
  const unsigned b_off = (unsigned)u * 512u + (unsigned)((bx & 1) * 16 + l16) * 16u;
  const unsigned t_base = (unsigned)(bx >> 1) * AA * t_pos;
  const bool busy = 4 * wave < a.ic2;          // wave-uniform
  v4i ra[D], rb[D];
  auto issue = [&](int k) {                    // k-th position in the order column by column
    const int p = A * (k % A) + k / A;
    buffer_load_cell(rw, a_off, p * w_pos, ra[k % D]);
    buffer_load_cell(rt, b_off, t_base + p * t_pos, rb[k % D]);
  };
  if (busy)
#pragma unroll
    for (int k = 0; k < D; ++k)
      if (k < AA) issue(k);
  for (int idx = tid; idx < 3 * AA * 4; idx += TB) {
    const int q = idx & 3, pa = idx >> 2;      // (array, position)
    *reinterpret_cast<float4 *>(&cst[0][0][0] + 4 * idx) =
        *reinterpret_cast<const float4 *>(a.scale + (long long)(pa / AA) * AA * a.ocpp + (long long)(pa % AA) * a.ocpp + by * 16 + 4 * q);
  }
  const bool adds = wave < 4;                  // wave-uniform
  const int ch = 4 * wave + (lane & 3), tl = lane >> 2;   // of a lane that adds up
  float m[AA];
#pragma unroll
  for (int i = 0; i < A; ++i) {
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const int k = A * i + r;
      v4i acc = {0, 0, 0, 0};
      if (busy) {
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ra[k % D], rb[k % D], acc, 0, 0, 0);
        if (k + D < AA) issue(k + D);
      }
      part[i & 1][r][wave][lane] = acc;
    }
    // the column's parts are in LDS; the column before the last has been added up, its place is free
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    if (adds) {
      const int *mine = reinterpret_cast<const int *>(&part[i & 1][0][0][0]) + wave * 64 + lane;
#pragma unroll
      for (int r = 0; r < A; ++r) {
        const int p = A * r + i;
        int s = __float_as_int(cst[2][p][ch]);
#pragma unroll
        for (int w = 0; w < NW; ++w) s += mine[(r * NW + w) * 256];
        m[p] = __builtin_fmaf((float)s, cst[0][p][ch], cst[1][p][ch]);
        asm volatile("" : "+v"(m[p]));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const int px = a.out_nhwc ? a.oc2 * 16 : 16;
  // element offset of pixel e of tile t of the block, or -1
  auto cell_of = [&](int tile, int e) -> long long {
    const int t = bx * 16 + tile;
    if (t >= a.t) return -1;
    const int n = t / a.nt, rem = t - n * a.nt, th = rem / a.wt, tw = rem - th * a.wt;
    const int oh = M * th + e / M, ow = M * tw + e % M;
    if (oh >= a.oh || ow >= a.ow) return -1;
    return (a.out_nhwc ? (long long)n * a.oh * a.ow * px + by * 16 : ((long long)n * a.oc2 + by) * a.oh * a.ow * 16) + ((long long)oh * a.ow + ow) * px;
  };
  v4i *cells = &part[A & 1][0][0][0];          // [tile][pixel], in the place of the column before the last
  if (adds) {
    const float bias = a.with_bias ? a.bias[by * 16 + ch] : 0.0f;
    const int at16 = tl * MM * 16 + ch;
    float y[MM];
    wino::tile_output<A>(m, y);
    if (a.out_type == EHIP_F32) {
      finish_channel_f32<A>(y, bias, a.with_bias != 0, a.with_relu != 0);
#pragma unroll
      for (int e = 0; e < MM; ++e) reinterpret_cast<float *>(cells)[at16 + 16 * e] = y[e];
    } else {
      unsigned pk[MM], old[MM];
#pragma unroll
      for (int e = 0; e < MM; ++e) {
        pk[e] = 0u;
        old[e] = 0u;
      }
      if (a.with_sum)
#pragma unroll
        for (int e = 0; e < MM; ++e) {
          const long long at = cell_of(tl, e);
          if (at >= 0) old[e] = static_cast<const uint8_t *>(a.out)[at + ch];
        }
      auto quantize = [&](auto out_c, auto relu_c, auto sum_c) {
        pack_channel<decltype(out_c)::value, A>(y, bias, 0, decltype(relu_c)::value, a.out_repS, a.out_z, decltype(sum_c)::value, old, pk);
      };
      auto relu_sum = [&](auto out_c) {
        if (a.with_sum) {
          if (a.with_relu) quantize(out_c, std::true_type{}, std::true_type{});
          else quantize(out_c, std::false_type{}, std::true_type{});
        } else {
          if (a.with_relu) quantize(out_c, std::true_type{}, std::false_type{});
          else quantize(out_c, std::false_type{}, std::false_type{});
        }
      };
      if (a.out_type == EHIP_U8) relu_sum(std::integral_constant<int, EHIP_U8>{});
      else relu_sum(std::integral_constant<int, EHIP_S8>{});
#pragma unroll
      for (int e = 0; e < MM; ++e) reinterpret_cast<uint8_t *>(cells)[at16 + 16 * e] = (uint8_t)pk[e];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
  if (a.out_type == EHIP_F32) {
    for (int c = tid; c < 64 * MM; c += TB) {
      const long long at = cell_of(c / (4 * MM), c / 4 % MM);
      if (at >= 0) *reinterpret_cast<v4i *>(static_cast<float *>(a.out) + at + 4 * (c & 3)) = cells[c];
    }
  } else {
    for (int c = tid; c < 16 * MM; c += TB) {
      const long long at = cell_of(c / MM, c % MM);
      if (at >= 0) *reinterpret_cast<v4i *>(static_cast<uint8_t *>(a.out) + at) = cells[c];
    }
  }
}

// Where it is the fastest form: while every workgroup has a CU of its own, with 129 to 512 input channels.  Fused stage with other
// tensors on every call, the form that ran before / this, us, at so many workgroups: tile size 6, 192 input channels 11.6 / 9.5 (112),
// 11.7 / 10.1 (256); 256 channels 13.4 / 10.1 (112), 13.7 / 10.9 (256); 384 channels 17.7 / 13.1 (128), 17.9 / 13.4 (224), 18.1 / 23.2 (320); 512 channels
// 20.4 / 14.7 (128), 20.4 / 15.8 (224), 21.6 / 28.2 (320); 128 channels 9.6 / 9.0 (112), but the layer as a whole 12.8 / 13.1 (208).  Tile size 5, 256
// channels 11.4 / 8.1 (208), 11.5 / 10.4 (304); 512 channels 15.3 / 10.9 (224), 15.6 / 19.5 (416).  Tile size 4, 256 channels 7.5 / 6.7 (208), 7.6 / 8.2 (400).
// (One block of tiles alone stays on the form that the tests of the choice pin for it: 20.0 / 14.7 with 512 channels.)
bool wino_split_applies(const WinoFusedArgs &a)
{
  const int A = a.tile ? a.tile : 6, nks = (a.ic2 + 3) / 4, blocks = (a.t + 15) / 16;
  if (nks > 8 || a.units_pad < 4 * nks || (a.out_type == EHIP_F32 && a.with_sum)) return false;
  if ((long long)A * A * a.units_pad * a.ocpp * 16 > 0x7fffffffll || (long long)((a.t + 31) / 32) * A * A * a.ic2 * 512 > 0x7fffffffll) return false;
  if (const char *env = getenv("EHIP_WINO_SPLIT")) return env[0] != '0';
  // (a switch that asks for one of the other forms)
  for (const char *k : {"EHIP_WINO_LANES", "EHIP_WINO_LANES_WRES", "EHIP_WINO_LANES_SLOTS", "EHIP_WINO_LANES_WAVES", "EHIP_WINO_RING"})
    if (getenv(k)) return false;
  return nks >= 3 && blocks >= 2 && (long long)blocks * a.oc2 <= 256;
}

hipError_t plan_wino_gemm_output_split(LaunchPlan &plan, const WinoFusedArgs &a0)
{
  WinoFusedArgs a = a0;
  const int A = a.tile ? a.tile : 6, nks = (a.ic2 + 3) / 4;
  a.nx = (a.t + 15) / 16;
  a.ny = a.oc2;
  const long long weights = (long long)a.units_pad * a.ocpp, tiles = (long long)(a.t + 31) / 32 * 32 * a.ic2;
  a.slots = weights > tiles;   // (what an XCD reads: an eighth of one and all of the other)
  const int grid = 8 * (a.slots ? (a.ny + 7) / 8 * a.nx : (a.nx + 7) / 8 * a.ny);
  void (*kernel)(const WinoFusedArgs *, void *, const float *) = nullptr;
#define EHIP_WS(A) kernel = nks <= 4 ? k_wino_gemm_output_lanes_split<A, 4> : k_wino_gemm_output_lanes_split<A, 8>
  if (A == 4) EHIP_WS(4);
  else if (A == 5) EHIP_WS(5);
  else EHIP_WS(6);
#undef EHIP_WS
  plan.name = "k_wino_gemm_output_lanes_split";
  return plan_set(plan, kernel, dim3(grid), dim3(nks <= 4 ? 256 : 512), 0, a, ArgBlock{}, ArgOut{a.out}, ArgBias{});
}

}  // namespace ehip
