// 1x1 layers with few output values: the K loop split over the waves of a workgroup.
//
// Replaces, for those layers, __execute_a160_s1 / _s2 and u8s8_gemm_kernel::op_gemm
// (src/elx_int8_conv_direct_1x1.cpp:234-480, src/kernel/elk_u8s8_gemm.hxx:66-406).
//
// Such a layer (one image: 512 -> 512 at 14 x 14 is 112 tiles of 32 x 32 results) is bound by the latency of one wave's chain:
// loads, K loop, epilogue.  The tiles that suit large layers (ehip_gemm1x1.hip) give 32 workgroups here, each of which pulls
// 100 KB through one CU and multiplies sixteen k-steps in a row.  In this kernel a workgroup owns ONE tile of 32 channels x
// 32 pixels and its NW waves take KPW k-steps (of 32 channels) each: all of a wave's operands are requested at once,
// straight into registers, so the chain is one trip to memory, KPW multiplies, one exchange of partial sums through LDS and
// the epilogue of 16 values per lane.  The last two are the first wave's alone: it adds up to eight partial sums and
// finishes the 32 x 32 values while the others have ended.
#include "ehip_internal.hpp"

namespace ehip {

// What every load of a wave needs -- operands AND per-channel constants: behind the argument structure (`rest`) the latter
// would be two more trips to memory one after the other -- as leading scalar arguments, preloaded with the wave.
// ny_rows = channel blocks | packed rows / 256 << 16; geom = stride_h | stride_w << 8 | dense << 16 | in_nhwc << 17 |
// out_nhwc << 18 | ic2 << 24; iow = iw | ow << 16; consts: [scale | shift | compensation][packed rows]
#define EHIP_SPLIT_HEAD                                                                                              \
  const uint8_t *in, const int8_t *w, const float *consts, const GemmArgs *rest, int p_total, int ohw, unsigned ohw_magic,  \
      int ihw, unsigned ny_rows, unsigned geom, unsigned iow, unsigned ow_magic, void *out

template <int NW, int KPW>
__global__ __launch_bounds__(64 * NW) void k_gemm1x1_split(EHIP_SPLIT_HEAD)
{
  __shared__ v4i part[(NW > 1 ? NW - 1 : 1) * 256];   // [wave - 1][quarter of the 16 results][lane]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  // (channel blocks next to each other: block b runs on XCD b % 8, so with a multiple of eight of them an XCD's L2 holds the
  // weights of its own ones only)
  const int ny = (int)(ny_rows & 0xffffu), ocpp = (int)(ny_rows >> 16) * kOcTile, iw = (int)(iow & 0xffffu), ow = (int)(iow >> 16);
  const int px = blockIdx.x / ny, oc0 = (blockIdx.x - px * ny) * 32;
  const int ic2 = (int)(geom >> 24), sh = (int)(geom & 0xffu), sw = (int)((geom >> 8) & 0xffu);
  const bool in_nhwc = (geom >> 17) & 1u, out_nhwc = (geom >> 18) & 1u, dense = (geom >> 16) & 1u;
  const int nks = (ic2 + 1) >> 1;
  const int ks0 = wave * KPW;

  int gp = px * 32 + l32;
  const bool valid = gp < p_total;
  gp = valid ? gp : p_total - 1;
  const int n = ohw == p_total ? 0 : fastdiv_any(gp, ohw, ohw_magic);
  const int r = gp - n * ohw;
  long long sp = r;
  if (!dense) {
    const int oh = fastdiv(r, ow, ow_magic);
    sp = (long long)(oh * sh) * iw + (r - oh * ow) * sw;
  }
  const uint8_t *src = in + (in_nhwc ? ((long long)n * ihw + sp) * ic2 * 16 : ((long long)n * ic2 * ihw + sp) * 16);
  const long long ustride = in_nhwc ? 16 : (long long)ihw * 16;
  v4i va[KPW], vb[KPW];
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int ks = ks0 + i < nks ? ks0 + i : nks - 1;
    int u = 2 * ks + lh;
    va[i] = *reinterpret_cast<const v4i *>(w + ((long long)u * ocpp + oc0 + l32) * 16);
    u = u < ic2 ? u : ic2 - 1;   // (an odd count's last unit multiplies zero weights)
    vb[i] = *reinterpret_cast<const v4i *>(src + u * ustride);
  }
  const int oc = oc0 + 16 * lh;
  OcConsts k;
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      k.sc[q] = *reinterpret_cast<const float4 *>(consts + oc + 4 * q);
      k.sh[q] = *reinterpret_cast<const float4 *>(consts + ocpp + oc + 4 * q);
      k.comp[q] = *reinterpret_cast<const v4i *>(consts + 2 * (size_t)ocpp + oc + 4 * q);
    }
  }
  GemmArgs a = load_args(rest);
  const int oc_real = a.oc2 * 16;
  v4i old;
  const size_t cell = out_nhwc ? (size_t)gp * oc_real + oc : (((size_t)n * a.oc2 + (oc >> 4)) * ohw + r) * 16;
  if (wave == 0 && a.ep.with_sum) old = *reinterpret_cast<const v4i *>(static_cast<const uint8_t *>(out) + (oc < oc_real ? cell : 0));
  v16i acc[1][1];
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[0][0][v] = 0;
#pragma unroll
  for (int i = 0; i < KPW; ++i)
    if (ks0 + i < nks)   // wave-uniform
      acc[0][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[i], vb[i] ^ (int)0x80808080, acc[0][0], 0, 0, 0);
  if (wave > 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      part[(wave - 1) * 256 + q * 64 + lane] = v4i{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]};
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v4i s = k.comp[q];
#pragma unroll
    for (int v = 1; v < NW; ++v) s += part[(v - 1) * 256 + q * 64 + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[0][0][4 * q + j] += s[j];
  }
  if (a.lean) {
    LeanConsts lk[1];
#pragma unroll
    for (int q = 0; q < 4; ++q) { lk[0].sc[q] = k.sc[q]; lk[0].sh[q] = k.sh[q]; }
    uint8_t *const cells[1] = {static_cast<uint8_t *>(out) + cell};
    const bool ok[1] = {valid};
    const v4i olds[1][1] = {{old}};
    lean_store<1, 1>(a.lean, a.ep, acc, lk, cells, ok, oc, oc_real, 0, olds);
    return;
  }
  // (blocked output here: the launcher sends nhwc output of these cases elsewhere)
  auto pixel_offset = [&](int p, bool &ok) -> size_t {
    ok = p < p_total;
    const int pc = ok ? p : 0;
    const int pn = ohw == p_total ? 0 : fastdiv_any(pc, ohw, ohw_magic);
    return ((size_t)pn * a.oc2 * ohw + (pc - pn * ohw)) * 16;
  };
  size_t pix[1], pixT[1][2];
  bool pvalid[1], validT[1][2];
  pix[0] = pixel_offset(px * 32 + l32, pvalid[0]);
  pixT[0][0] = pixel_offset(px * 32 + (lane >> 2), validT[0][0]);
  pixT[0][1] = pixel_offset(px * 32 + (lane >> 2) + 16, validT[0][1]);
  // (the partial sums have been read: their first 4 KB are the exchange patch of 4-byte outputs)
  epilogue_wave<1, 1, false, true>(a.ep, acc, k, oc, oc, pix, pvalid, oc_real, (size_t)ohw * 16, out,
                                   a.ep.out_type == EHIP_F32 || a.ep.out_type == EHIP_S32 ? part : nullptr, pixT, validT);
}

namespace {
typedef void (*split_kernel_t)(EHIP_SPLIT_HEAD);
split_kernel_t split_kernel(int nks, int &nw)
{
  nw = nks <= 1 ? 1 : (nks <= 2 ? 2 : (nks <= 16 ? 4 : 8));
  if (nks <= 1) return k_gemm1x1_split<1, 1>;
  if (nks <= 2) return k_gemm1x1_split<2, 1>;
  if (nks <= 4) return k_gemm1x1_split<4, 1>;
  if (nks <= 8) return k_gemm1x1_split<4, 2>;
  if (nks <= 12) return k_gemm1x1_split<4, 3>;
  if (nks <= 16) return k_gemm1x1_split<4, 4>;
  return nks <= 32 ? k_gemm1x1_split<8, 4> : k_gemm1x1_split<8, 8>;
}
}  // namespace

bool gemm1x1_split_applies(const GemmArgs &a, int nbatch)
{
  if (nbatch != 1 || a.kh * a.kw > 1 || a.ep.shift_tab || a.ic2 > 128) return false;
  if (a.stride_h > 255 || a.stride_w > 255 || a.iw >= 65536 || a.ow >= 65536 || a.oc2 >= 65536) return false;
  // (scale, shift and compensation in one allocation)
  if (a.ep.shift != a.ep.scale + a.ocpp || reinterpret_cast<const float *>(a.ep.comp) != a.ep.scale + 2 * (size_t)a.ocpp) return false;
  if (a.out_nhwc && !lean_mode(a.ep, false)) return false;
  for (const char *other : {"EHIP_GEMM1X1_RES", "EHIP_GEMM1X1_WRES", "EHIP_GEMM_VARIANT", "EHIP_GEMM_SMALLK"})   // (another kernel asked for)
    if (const char *env = getenv(other)) if (env[0]) return false;
  if (const char *env = getenv("EHIP_GEMM1X1_SPLIT")) return env[0] != '0';
  // Up to three workgroups per CU with 65-512 input channels, more with fewer (whose workgroups are smaller), fewer with more
  // (whose own workgroups elsewhere share the operands better).  Kernel time, other kernels / this one, us:
  //   32 -> 64 at 112 x 112:    N = 1 (784 tiles) 3.4 / 3.0, N = 2 3.6 / 3.4, N = 4 (3136) 3.9 / 4.3
  //   64 -> 128 at 56 x 56:     N = 1 (392) 4.3 / 2.9, N = 4 (1568) 4.4 / 3.5, N = 8 4.6 / 4.7
  //   128 -> 128 at 56 x 56:    N = 2 (784) 3.8 / 3.4, N = 4 (1568) 4.0 / 4.3
  //   512 -> 512 at 14 x 14:    N = 1 (112) 3.7 / 3.0, N = 8 (784) 4.6 / 4.1, N = 16 (1568) 4.9 / 5.8
  //   1024 -> 1024 at 7 x 7:    N = 1 (64) 5.2 / 3.2, N = 8 (416) 6.2 / 4.3, N = 16 (800) 5.8 / 5.8
  //   2048 -> 512 at 7 x 7:     N = 1 (32) 8.4 / 3.6, N = 16 (400) 9.8 / 6.6, N = 32 (784) 10.2 / 10.8
  const int nks = (a.ic2 + 1) / 2;
  const long long tiles = (long long)((a.p_total + 31) / 32) * ((a.oc2 * 16 + 31) / 32);
  return tiles <= (nks <= 2 ? 1600 : (nks <= 16 ? 900 : 640));
}

hipError_t plan_gemm1x1_split(LaunchPlan &plan, const GemmArgs &a0)
{
  GemmArgs a = a0;
  a.lean = lean_mode(a.ep, false);
  int nw = 0;
  const split_kernel_t kernel = split_kernel((a.ic2 + 1) / 2, nw);
  a.nx = (a.p_total + 31) / 32;
  a.ny = (a.oc2 * 16 + 31) / 32;
  const bool dense = a.stride_h == 1 && a.stride_w == 1 && a.iw == a.ow;
  const unsigned geom = (unsigned)a.stride_h | (unsigned)a.stride_w << 8 | (dense ? 1u << 16 : 0u) | (a.in_nhwc ? 1u << 17 : 0u) |
      (a.out_nhwc ? 1u << 18 : 0u) | (unsigned)a.ic2 << 24;
  plan.name = "k_gemm1x1_split";
  return plan_set(plan, kernel, dim3((unsigned)(a.nx * a.ny)), dim3(64 * nw), 0, a, ArgIn{a.in}, a.w, a.ep.scale, ArgBlock{}, a.p_total,
                  a.ohw, a.ohw_magic, a.ihw, (unsigned)a.ny | (unsigned)(a.ocpp / kOcTile) << 16, geom,
                  (unsigned)a.iw | (unsigned)a.ow << 16, a.ow_magic, ArgOut{a.out});
}

}  // namespace ehip
