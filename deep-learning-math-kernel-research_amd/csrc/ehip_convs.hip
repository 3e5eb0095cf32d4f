// k x k direct convolutions as a GEMM over [tap][unit] with few output values: the K loop shared out among the waves of a
// workgroup.
//
// Replaces, for those layers, elx_int8_conv_direct_t::conv_a160 + gemm_a160 and the u8s8 GEMM micro-kernel
// (src/elx_int8_conv_direct.cpp:227-423, src/kernel/elk_u8s8_gemm.hxx:66-406).
#include "ehip_internal.hpp"
#include "ehip_convs_at.hpp"
#include "ehip_wino_input.hpp"

namespace ehip {

// Such a layer is bound by one workgroup's chain: 64 x 64 results walk K = taps x channels in fills of 64 to 128 that pass the LDS with
// a barrier each, 0.11 us a step of 32 (7x7, 480 -> 16 at 34 x 34, N = 2: 735 steps, 83 us, on 37 CUs).  Here the eight waves of a
// workgroup take an eighth of the steps each, with their operands straight from memory six to ten steps ahead, no barrier and
// no LDS until the sums meet: the chain is an eighth, and what is left is the stream into a CU (2 KB a step: 735 steps 15 us, 98 GB/s; loads alone get 115 from the L2).  A tap is
// the same for a wave's lanes, so the pixels' addresses are worked out once per tap and a step adds a scalar.  Taps outside the
// image are read past the end of the buffer, which gives code 0 as the padding does.  The sums are integers: exact in any order.
// us, with other tensors in turn: that layer 83.1 -> 19.1; 7x7 380 -> 256 at 14 x 14, N = 4 84.0 -> 14.5; 5x5 s2 160 -> 32 at 14 x 14, N = 5 21.3 -> 6.4; 5x5 256 ->
// 256 at 14 x 14, N = 8 23.6 -> 10.0; 3x3 512 -> 64 at 28 x 28, N = 4 (the 3x3 kernel) 15.8 -> 7.2.
// Workgroup = 32 TM channels x 32 TN pixels, a wave = every NW-th part of the K loop.  a.nx = pixel blocks, a.ny = channel blocks.
template <int TM, int TN, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_gemm_u8s8_split(const GemmArgs *rest, const uint8_t *in, void *out)
{
  GemmArgs a = load_args(rest);
  a.in = in; a.out = out;
  constexpr int T = TM * TN, D = T == 1 ? 10 : (T == 2 ? 8 : (T == 4 ? 6 : 3));   // tiles; k-steps in flight
  constexpr int PW = T <= 4 ? NW : NW / 2;   // waves whose sums fit the LDS at once
  extern __shared__ v4i part[];        // [wave][tile][quarter of the 16 results][lane]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int bx = blockIdx.x / a.ny, oc0 = (blockIdx.x - bx * a.ny) * 32 * TM;
  const int pix0 = bx * 32 * TN;
  // ---- the lane's pixels: input row and column of the first tap, byte of the image and unit -----------------------
  const SplitStrides strides = split_strides(a.in_nhwc != 0, a.ic2, a.ihw);
  int ihb[TN], iwb[TN];
  unsigned base[TN];
#pragma unroll
  for (int nt = 0; nt < TN; ++nt) {
    int gp = pix0 + 32 * nt + l32;
    gp = gp < a.p_total ? gp : a.p_total - 1;
    const int n = a.ohw == a.p_total ? 0 : fastdiv_any(gp, a.ohw, a.ohw_magic);
    const int r = gp - n * a.ohw, oh = fastdiv(r, a.ow, a.ow_magic);
    ihb[nt] = oh * a.stride_h - a.pad_t;
    iwb[nt] = (r - oh * a.ow) * a.stride_w - a.pad_l;
    base[nt] = split_image(strides, n, lh, a.ic2, a.ihw);
  }
  const int images = (a.p_total + a.ohw - 1) / a.ohw;
  const BufferRsrc rin = make_rsrc(a.in, (unsigned)images * a.ic2 * a.ihw * 16u);
  const BufferRsrc rw = make_rsrc(a.w, (unsigned)a.k_real * a.ocpp * 16u);
  unsigned aoff[TM];
#pragma unroll
  for (int mt = 0; mt < TM; ++mt) aoff[mt] = (unsigned)(lh * a.ocpp + oc0 + 32 * mt + l32) * 16u;
  // ---- the wave's k-steps: pairs of units, tap by tap ---------------------------------------------------------------
  const int P = (a.ic2 + 1) >> 1, S = a.kh * a.kw * P;
  const int s0 = S * wave / NW, s1 = S * (wave + 1) / NW;
  int si = s0, tap = s0 / P, pr = s0 - tap * P;
  unsigned voff[TN];
  auto at_tap = [&]() {
    const int kr = tap / a.kw, kc = tap - kr * a.kw;
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) voff[nt] = split_tap(strides, base[nt], ihb[nt] + kr, iwb[nt] + kc, a.ih, a.iw);
  };
  at_tap();
  v4i ra[D][TM], rb[D][TN];
  auto issue = [&](int slot) {
    const bool live = si < s1;
    const int units = live ? a.ic2 : 0;   // (past the last step every lane is past the buffers)
    const unsigned wat = (unsigned)(tap * a.units_pad + 2 * pr) * (unsigned)a.ocpp * 16u, iat = split_step(strides, pr);   // scalar
#pragma unroll
    for (int mt = 0; mt < TM; ++mt) buffer_load_cell(rw, split_lane(aoff[mt], pr, lh, units), live ? wat : 0u, ra[slot][mt]);
#pragma unroll
    for (int nt = 0; nt < TN; ++nt) buffer_load_cell(rin, split_lane(voff[nt], pr, lh, units), live ? iat : 0u, rb[slot][nt]);
    ++si;
    if (++pr == P) {
      pr = 0;
      ++tap;
      at_tap();
    }
  };
#pragma unroll
  for (int k = 0; k < D; ++k) {
    issue(k);
    __builtin_amdgcn_sched_barrier(0);
  }
  v16i acc[TM][TN];
#pragma unroll
  for (int mt = 0; mt < TM; ++mt)
#pragma unroll
    for (int nt = 0; nt < TN; ++nt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mt][nt][v] = 0;
#pragma unroll 1
  for (int s = s0; s < s1; s += D) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
#pragma unroll
      for (int nt = 0; nt < TN; ++nt) {
        const v4i b = rb[k][nt] ^ (int)0x80808080;
#pragma unroll
        for (int mt = 0; mt < TM; ++mt) acc[mt][nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ra[k][mt], b, acc[mt][nt], 0, 0, 0);
      }
      issue(k);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // ---- the parts meet in LDS; a wave finishes a tile ------------------------------------------------------------------
  auto leave = [&](int at) {
#pragma unroll
    for (int mt = 0; mt < TM; ++mt)
#pragma unroll
      for (int nt = 0; nt < TN; ++nt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          part[((at * T + mt * TN + nt) * 4 + q) * 64 + lane] =
              v4i{acc[mt][nt][4 * q], acc[mt][nt][4 * q + 1], acc[mt][nt][4 * q + 2], acc[mt][nt][4 * q + 3]};
  };
  if constexpr (PW < NW) {             // the upper half's sums first, into the lower half's
    if (wave >= PW) leave(wave - PW);
    __syncthreads();
    if (wave < PW)
#pragma unroll
      for (int mt = 0; mt < TM; ++mt)
#pragma unroll
        for (int nt = 0; nt < TN; ++nt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const v4i x = part[((wave * T + mt * TN + nt) * 4 + q) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[mt][nt][4 * q + j] += x[j];
          }
    __syncthreads();
    if (wave < PW) leave(wave);
  } else leave(wave);
  __syncthreads();
  if (wave >= T) return;
  const int oc_real = a.oc2 * 16, oc = oc0 + 32 * (wave / TN) + 16 * lh, p0 = pix0 + 32 * (wave % TN);
  OcConsts k0;
  load_consts(k0, a.ep, oc);
  v16i sum[1][1];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v4i s = k0.comp[q];
#pragma unroll
    for (int w = 0; w < PW; ++w) s += part[((w * T + wave) * 4 + q) * 64 + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[0][0][4 * q + j] = s[j];
  }
  // element offset of output pixel gp's cell in 16-channel block 0 (nhwc: its channel vector)
  auto pixel_offset = [&](int gp, bool &valid) -> size_t {
    valid = gp < a.p_total;
    const int gpc = valid ? gp : 0;
    if (a.out_nhwc) return (size_t)gpc * oc_real;
    const int n = a.ohw == a.p_total ? 0 : fastdiv_any(gpc, a.ohw, a.ohw_magic);
    return ((size_t)n * a.oc2 * a.ohw + (gpc - n * a.ohw)) * 16;
  };
  size_t pix[1], pixT[1][2];
  bool pvalid[1], validT[1][2];
  int cls[1] = {0};
  if (a.ep.shift_tab) {                // border class of the lane's pixel
    int gp = p0 + l32;
    gp = gp < a.p_total ? gp : a.p_total - 1;
    const int r = gp - (a.ohw == a.p_total ? 0 : fastdiv_any(gp, a.ohw, a.ohw_magic)) * a.ohw;
    const int oh = fastdiv(r, a.ow, a.ow_magic);
    cls[0] = a.cls_h[oh] * a.ncls_w + a.cls_w[r - oh * a.ow];
  }
  pix[0] = pixel_offset(p0 + l32, pvalid[0]);
  pixT[0][0] = pixel_offset(p0 + (lane >> 2), validT[0][0]);
  pixT[0][1] = pixel_offset(p0 + (lane >> 2) + 16, validT[0][1]);
  // (4-byte outputs: the wave's tile of the first wave's parts, which it has read, is the exchange patch)
  v4i *xlds = (a.ep.out_type == EHIP_F32 || a.ep.out_type == EHIP_S32) && !a.out_nhwc ? part + wave * 256 : nullptr;
  epilogue_wave<1, 1, true, true>(a.ep, sum, k0, oc, oc, pix, pvalid, oc_real, a.out_nhwc ? (size_t)16 : (size_t)a.ohw * 16, a.out, xlds,
                                  pixT, validT, cls);
}

// The form for a layer: 0, 1, 2, 3, 4 = 32 x 32, 32 x 64, 64 x 64, 32 x 128, 64 x 128 channels x pixels a workgroup, -1 = none.  The smallest whose workgroups have
// a CU of their own; a second round costs what the first did.  The kernel that ran before / the three forms, us, by units of 16
// channels of all taps:
//   instead of the general kernel (nhwc input, 5x5 or 7x7, zero points): 36 units 5.3 / 5.6 6.1 6.6 (98 workgroups of 32 x 32); 50 7.5 / 6.8 7.3 7.4 (98); 72 7.6 / 10.3 7.5 7.6
//     (490), 7.8 / 19.8 13.7 7.9 (980); 100 10.7 / 10.1 6.6 8.0 (490), 10.9 / 18.8 11.9 8.3 (980), 12.7 / 31.7 21.9 14.8 (1568); 144 11.6 / 12.3 10.1 10.2 (490), 11.7 / 23.0
//     20.0 10.7 (980), 14.4 / 37.5 35.6 19.7 (1568)
//   instead of the 3x3 kernel: 72 units 4.7 / 5.3 6.0 6.4 (98); 144 6.7 / 5.3 7.3 7.7 (98), 5.8 / 9.3 7.4 7.7 (490), 8.2 / 17.2 13.5 8.1 (980); 288 15.8 / 7.2 8.7 9.0 (196), 10.0 / 11.5 8.9
//     9.3 (490), 13.6 / 23.1 18.0 11.1 (980); stride 2, 288 13.1 / 6.5 9.0 9.4 (32), 15.1 / 29.1 25.5 15.6 (980)
// and 32 x 128 and 64 x 128 with 31360 pixels, 32 and 64 channels: the general kernel 72 units 9.1 / 10.0, 9.2 / 11.7; 100 12.4 / 10.2, 12.5 / 11.2; 3x3, 144 14.5 / 15.1,
// 15.3 / 16.3; 7x7, 196 21.6 / 12.9, 21.9 / 15.0; 5x5, 200 20.1 / 18.0, 20.5 / 19.9; the 3x3 kernel 144 8.8 / 9.9, 14.0 / 11.4 (7840 and 256 channels 11.1 / 11.3); 288
// 16.2 / 13.3, 26.7 / 16.6.
// (50 units, blocked input: 7.0 / 7.1 and 7.2 with 98 to 245 workgroups, hence 64 there.)
// The 3x3 kernel, stride 1, is at its best where its workgroups come to one round, no wave is without channels or shares its own
// with another, and one fill of the LDS holds all input channels (up to 512: 288 units).  There it takes less for more pixels, because it
// reads them once for 128 channels, where a workgroup here has 32 or 64.  427 layers of 128 to 1024 input channels, 3x3 kernel / the form:
//   32 x 64, 288 units, more than 2048 pixels: 9.8 / 9.7 to 10.4 (up to 2048: 9.7 to 10.7 / 8.7 to 9.1; 216 units 8.1 to 8.3 / 7.5 to 8.0);
//   64 x 64: 216 units 8.1 to 8.8 / 9.1 to 10.1; 288 units, more than 2048 pixels 10.0 to 10.8 / 10.4 to 10.8 (up to 2048: 9.9 to 10.7 / 9.2 to 9.5);
//   32 x 128, 32 channels: 216 units 11.3 to 12.0 / 11.5 to 11.9; 288 units 12.9 / 12.9 to 13.5;
//   64 x 128: 512 -> 512 at 7 x 7, N = 64 11.6 to 14.1 / 15.4 (it moves with the box and its clock, this kernel does not); 384 -> 512 there
//     9.3 to 10.9 / 13.3; 768 21.1 to 24.6 / 19.3 to 19.6, 1024 21.8 to 25.3 / 23.5.
// Two rounds of it still beat 32 x 128 and 64 x 128 (216 units 10.9 to 13.4 / 12.3 to 13.3, 288 14.2 to 17.1 / 14.9 to 15.7), not 64 x 64 (13.8 /
// 11.0); nor do three (384 -> 192 at 14 x 14, N = 48, 18.8 / 14.8; 512 -> 512 at 14 x 14, N = 20 22.5 to 23.7 / 15.7 to 17.6).  With more
// channels it fills twice (432 units, one round: 18.0 / 11.8 to 15.0), with half of the waves idle (64 channels) it takes 15 to 19 us for 10
// to 16, with wide rows 14 to 17 for 8 to 16.
int conv_split_pick(const GemmArgs &a, int nbatch, const Conv3x3Tiles *planes)
{
  const int taps = a.kh * a.kw;
  if (nbatch != 1 || taps <= 1 || taps > 64 || a.ep.with_sum) return -1;
  if (planes && (a.pad_t > 255 || a.pad_l > 255)) return -1;   // (what the 3x3 kernel refuses)
  const long long in_bytes = (long long)(a.p_total / a.ohw) * a.ic2 * a.ihw * 16, w_bytes = (long long)taps * a.units_pad * a.ocpp * 16;
  if (in_bytes > 0x7fffffffll || w_bytes > 0x7fffffffll) return -1;
  if (const char *env = getenv("EHIP_CONV_SPLIT")) return env[0] >= '0' && env[0] <= '4' ? env[0] - '0' : -1;
  // (another kernel asked for)
  for (const char *other : {"EHIP_GEMM_VARIANT", "EHIP_GEMM_SMALLK", "EHIP_CONV3X3V_VARIANT", "EHIP_CONV3X3V_UNROLL", "EHIP_CONV3X3V_SPLIT_LAST",
                            "EHIP_CONV3X3V_SHARED"})
    if (const char *env = getenv(other)) if (env[0]) return -1;
  const int units = taps * a.ic2;
  const long long px32 = (a.p_total + 31) / 32, px64 = (a.p_total + 63) / 64, oc32 = (a.oc2 + 1) / 2, oc64 = (a.oc2 + 3) / 4;
  const bool apart = planes && a.stride_h == 1 && planes->apart && 32 * a.oc2 > planes->channels, best = apart && units <= 288;   // (see above)
  const bool one = best && planes->count <= 256;
  if (px32 * oc32 <= 256) return units >= (planes ? 128 : a.in_nhwc ? 40 : 64) ? 0 : -1;
  if (px64 * oc32 <= 256) {
    if (one && units >= 256 && a.p_total > 2048 && planes->channels == 128) return -1;
    return units >= (planes ? 216 : 64) ? 1 : -1;
  }
  if (planes && a.stride_h > 1) return -1;
  const long long px128 = (a.p_total + 127) / 128;
  if (units < (planes ? 216 : 96)) return -1;
  if (px64 * oc64 <= 256) return one && (units < 256 || a.p_total > 2048) ? -1 : 2;
  if (best && planes->count <= 512) return -1;
  if (px128 * oc32 <= 256) return 3;
  return px128 * oc64 <= 256 && (planes ? !(apart && planes->count <= 256) : taps > 9) ? 4 : -1;
}

hipError_t plan_conv_split(LaunchPlan &plan, const GemmArgs &a0, int form)
{
  GemmArgs a = a0;
  a.k_real = a.kh * a.kw * a.units_pad;
  const int tm = form == 2 || form == 4 ? 2 : 1, tn = form >= 3 ? 4 : (form >= 1 ? 2 : 1);
  a.nx = (a.p_total + 32 * tn - 1) / (32 * tn);
  a.ny = (a.oc2 * 16 + 32 * tm - 1) / (32 * tm);
  void (*kernel)(const GemmArgs *, const uint8_t *, void *) =
      form == 0 ? k_gemm_u8s8_split<1, 1, 8> : form == 1 ? k_gemm_u8s8_split<1, 2, 8> : form == 2 ? k_gemm_u8s8_split<2, 2, 8> :
      form == 3 ? k_gemm_u8s8_split<1, 4, 8> : k_gemm_u8s8_split<2, 4, 8>;
  // (channels, pixels of a workgroup)
  static const char *const names[] = {"k_gemm_u8s8_split<32,32>", "k_gemm_u8s8_split<32,64>", "k_gemm_u8s8_split<64,64>", "k_gemm_u8s8_split<32,128>",
                                      "k_gemm_u8s8_split<64,128>"};
  plan.name = names[form];
  return plan_set(plan, kernel, dim3((unsigned)(a.nx * a.ny)), dim3(512), (size_t)(tm * tn > 4 ? 4 : 8) * tm * tn * 4096, a, ArgBlock{}, ArgIn{a.in}, ArgOut{a.out});
}

}  // namespace ehip
