// Winograd GEMMs + output transform for layers of about one round of workgroups: the columns of the positions shared out among the
// waves of a workgroup.
//
// Replaces, for those layers, elx_int8_conv_wino_gemm_t::execute + trans_output as the reference's fused schedule
// runs them per thread (a161, src/elx_int8_conv_wino_xopt.hpp:21-179; src/elx_int8_conv_wino_gemm.cpp:23-205,
// src/elx_conv_wino_trans_output.cpp:212-423).
//
// Compiled with the accumulators in the ordinary vector registers, like ehip_wino_lanes.hip.
#include "ehip_wino_pack.hpp"
#include <type_traits>

namespace ehip {

// A layer of few tiles is bound by the chain of one wave: with the weights of 16 channels resident in LDS a wave takes its tiles
// through all A x A positions one after the other, alone on its SIMD (5.5 clocks an instruction) behind the 147 KB of weights that
// the workgroup waits for first; through the ring, every k-step of every position passes a barrier and the LDS.  Here the
// positions themselves are shared out: a wave takes one column of them, A positions, over all input channels -- a sixth of the
// chain, no barrier and no LDS before the column is whole, and so few accumulators that two k-steps of all A positions are in flight
// (24 to 36 loads of 1 KB a wave).  The column is requantized and taken through the first dimension of the output transform where
// it is; what is left of it (A - 2 values) meets the other columns in LDS, and the waves share the rows of the output.  Tile
// size 4, a two-dimensional formula in the reference, meets as positions.
// The bytes through the L1 of a CU are what is left: 3 KB for two matrix instructions with 32 channels x 16 tiles a workgroup, 885 KB a CU
// for 512 -> 512, 256 tiles (15.8 us; the 115 GB/s that a CU gets from its L2 while all of them read would be 7.7).  Both halves of a group of 32 packed rows
// belong to a workgroup of 32 channels, because a half alone uses half of every cache line: 16.7 against 18.4 us for 16 channels x 32
// tiles, of the same bytes.  An XCD takes neighbouring groups of channels, not every eighth, for the same reason (13.3 / 12.6).
// Tried: two k-steps less ahead by the compiler's order of the first loads (17.6 against 15.8: hence the scheduling barriers), twelve
// waves of two blocks of tiles (24.8 against 19.3 with six of them), 16 channels x 64 tiles (15.6 against 13.4 us of 32 x 32).
// Workgroup = 16 RO channels x 16 RT tiles, a wave = a column of their positions.  a.nx = groups of RT blocks of 16 tiles, a.ny =
// groups of 16 RO channels; an XCD takes every 2^a.slots-th group of
// tiles of a run of channels.
template <int A, int RO, int RT>
__global__ __launch_bounds__(64 * A, A == 4 ? 1 : 2) void k_wino_gemm_output_lanes_cols(const WinoFusedArgs *rest, void *out, const float *bias_)
{
  WinoFusedArgs a = load_args(rest);
  a.out = out; a.bias = bias_;
  constexpr int AA = A * A, M = A - 2;
  constexpr int RV = A == 4 ? A : M;           // values of a column that the second dimension takes
  constexpr int TASKS = A == 4 ? 1 : M;        // of a block of tiles x 16 channels
  constexpr int UN = A == 4 ? (RO * RT == 1 ? 4 : 2) : (RO * RT == 4 ? 1 : 2);   // k-steps in flight
  extern __shared__ float4 lds[];              // [block][value][column][lane], then a wave's constants [3][A][4 RO]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int col = wave;                        // the wave's column of the positions
  // (the grid's first dimension is a multiple of eight: a workgroup's XCD is its number there modulo eight)
  const int xcd = blockIdx.x & 7, xa = a.slots;   // xa: log2 of the XCDs beside each other along the tiles
  const int bx = ((int)(blockIdx.x >> 3) << xa) + (xcd & ((1 << xa) - 1)), by = (xcd >> xa) * (int)gridDim.y + (int)blockIdx.y;
  if (bx >= a.nx || by >= a.ny) return;        // whole workgroup
  // ---- a column's constants, the wave's own ---------------------------------------------------------------------
  constexpr int NQ = 4 * RO, NC = 3 * A * NQ;                // cells
  float4 *cst = lds + RO * RT * RV * A * 64 + wave * NC;
  auto const_cell = [&](int j) {               // (past the end the last cell once more: the same bytes)
    const int idx = lane + 64 * j;
    return idx < NC ? idx : NC - 1;
  };
  auto load_const = [&](int j) {
    const int idx = const_cell(j), q = idx % NQ, r = idx / NQ % A, arr = idx / NQ / A;
    return *reinterpret_cast<const float4 *>(a.scale + ((long long)arr * AA + A * r + col) * a.ocpp + by * (16 * RO) + 4 * q);
  };
  static_assert(NC <= 192, "three cells a lane");
  const float4 c0 = load_const(0), c1 = load_const(1), c2 = load_const(NC > 128 ? 2 : 1);
  // ---- operands: straight from memory, UN k-steps of the column ahead -------------------------------------------
  // the workgroup's 16 channels are one block of the output: of the group of 32 packed rows (row 8 gq + 4 h + j holds channel
  // 16 h + 4 gq + j) the rows of half h
  const unsigned w_pos = (unsigned)a.units_pad * (unsigned)a.ocpp * 16u, t_pos = (unsigned)a.ic2 * 512u;   // bytes (the launcher
  const unsigned nblk = (unsigned)((a.t + 31) >> 5);
  const BufferRsrc rw = make_rsrc(a.w, AA * w_pos), rt = make_rsrc(a.tin, nblk * AA * t_pos);              // checks 32 bits)
  const unsigned w_ks = (unsigned)a.ocpp * 64u;
  const unsigned a_off = (unsigned)(g * a.ocpp + (RO == 2 ? by * 32 + l16 : (by >> 1) * 32 + (by & 1) * 4 + 8 * (l16 >> 2) + (l16 & 3))) * 16u;
  unsigned b_off[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    const unsigned b = (unsigned)(bx * RT + j);   // (a block past the last one: past the buffer, zeros)
    b_off[j] = (b >> 1) * AA * t_pos + (unsigned)g * 512u + (b & 1) * 256u + (unsigned)l16 * 16u;
    b_off[j] = (b >> 1) < nblk ? b_off[j] : 0x80000000u;
  }
  const int nks = (a.ic2 + 3) >> 2;
  v4i ra[UN][A][RO], rb[UN][A][RT];
  auto issue = [&](int slot, int r, int ks) {
    // (k-steps and units past the last one: past the buffer, zeros)
    const bool in = ks < nks;
    const unsigned wo = in ? a_off + (unsigned)ks * w_ks : 0x80000000u;
#pragma unroll
    for (int h = 0; h < RO; ++h) buffer_load_cell(rw, wo + 256u * h, (unsigned)(A * r + col) * w_pos, ra[slot][r][h]);
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const unsigned to = 4 * ks + g < a.ic2 ? b_off[j] + (unsigned)ks * 2048u : 0x80000000u;
      buffer_load_cell(rt, to, (unsigned)(A * r + col) * t_pos, rb[slot][r][j]);
    }
  };
#pragma unroll
  for (int s = 0; s < UN; ++s)
#pragma unroll
    for (int r = 0; r < A; ++r) {
      issue(s, r, s);
      __builtin_amdgcn_sched_barrier(0);       // (in the loop's order, or its waits are for more than they need)
    }
  cst[const_cell(0)] = c0;
  cst[const_cell(1)] = c1;
  if (NC > 128) cst[const_cell(2)] = c2;
  v4i acc[A][RO * RT];
#pragma unroll
  for (int r = 0; r < A; ++r)
#pragma unroll
    for (int j = 0; j < RO * RT; ++j) acc[r][j] = v4i{0, 0, 0, 0};
#pragma unroll 1
  for (int ks = 0; ks < nks; ks += UN) {
#pragma unroll
    for (int s = 0; s < UN; ++s)
#pragma unroll
      for (int r = 0; r < A; ++r) {
#pragma unroll
        for (int j = 0; j < RO * RT; ++j) acc[r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ra[s][r][j / RT], rb[s][r][j % RT], acc[r][j], 0, 0, 0);
        issue(s, r, ks + s + UN);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  // ---- the column requantized and taken through the first dimension of the output transform ---------------------
#pragma unroll
  for (int j = 0; j < RO * RT; ++j) {
    float f[4][A];
    // the quad of channels that the lane holds, and the half of them that it is in
    const int h = RO == 2 ? g & 1 : 0, gq = RO == 2 ? 2 * (j / RT) + (g >> 1) : g, q = 4 * h + gq;
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const float4 sc = cst[r * NQ + q], sh = cst[(A + r) * NQ + q], cf = cst[(2 * A + r) * NQ + q];
      f[0][r] = __builtin_fmaf((float)(acc[r][j][0] + __float_as_int(cf.x)), sc.x, sh.x);
      f[1][r] = __builtin_fmaf((float)(acc[r][j][1] + __float_as_int(cf.y)), sc.y, sh.y);
      f[2][r] = __builtin_fmaf((float)(acc[r][j][2] + __float_as_int(cf.z)), sc.z, sh.z);
      f[3][r] = __builtin_fmaf((float)(acc[r][j][3] + __float_as_int(cf.w)), sc.w, sh.w);
    }
    float o[4][RV];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (A == 4) {                  // (a two-dimensional formula in the reference: the positions themselves)
#pragma unroll
        for (int r = 0; r < A; ++r) o[k][r] = f[k][r];
      } else out_1d<A>(f[k], o[k]);
    }
#pragma unroll
    for (int r = 0; r < RV; ++r)
      lds[(((h * RT + j % RT) * RV + r) * A + col) * 64 + 16 * gq + l16] = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
  }
  __syncthreads();
  // ---- the second dimension: a wave per block of tiles and row of the output -------------------------------------
  const int px = a.out_nhwc ? a.oc2 * 16 : 16;
#pragma unroll 1
  for (int task = wave; task < RO * RT * TASKS; task += A) {
    const int cb = task / TASKS, r0 = task % TASKS;   // (channel half, block of tiles), row of the output
    const int by16 = RO * by + cb / RT;
    if (by16 >= a.oc2) break;                    // (an odd last half)
    const int t = (bx * RT + cb % RT) * 16 + l16;
    const bool valid = t < a.t;
    float4 bias = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.with_bias) bias = *reinterpret_cast<const float4 *>(a.bias + by16 * 16 + 4 * g);
    const int tc = valid ? t : 0;
    const int n = tc / a.nt, rem = tc - n * a.nt, th = rem / a.wt, tw = rem - th * a.wt;
    const size_t plane = a.out_nhwc ? (size_t)n * a.oh * a.ow * px + by16 * 16 : ((size_t)n * a.oc2 + by16) * a.oh * a.ow * 16;
    constexpr int ROWS = M / TASKS, PX = ROWS * M;   // pixels of a task
    float y[4][PX];
    if constexpr (A == 4) {
      float f[4][AA];
#pragma unroll
      for (int p = 0; p < AA; ++p) {
        const float4 v = lds[(cb * AA + p) * 64 + lane];
        f[0][p] = v.x; f[1][p] = v.y; f[2][p] = v.z; f[3][p] = v.w;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) wino::tile_output<4>(f[k], y[k]);
    } else {
      float f[4][A];
#pragma unroll
      for (int i = 0; i < A; ++i) {
        const float4 v = lds[((cb * M + r0) * A + i) * 64 + lane];
        f[0][i] = v.x; f[1][i] = v.y; f[2][i] = v.z; f[3][i] = v.w;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) out_1d<A>(f[k], y[k]);
    }
    if (a.out_type == EHIP_F32) {
#pragma unroll
      for (int e = 0; e < PX; ++e) {
        typedef float v4f __attribute__((ext_vector_type(4)));
        v4f vv;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float x = y[k][e];
          if (a.with_bias) x = x + comp_of(bias, k);
          if (a.with_relu) x = x > 0.0f ? x : 0.0f;
          vv[k] = x;
        }
        const int oh = M * th + r0 + e / M, ow = M * tw + e % M;
        if (valid && oh < a.oh && ow < a.ow)
          __builtin_nontemporal_store(vv, reinterpret_cast<v4f *>(static_cast<float *>(a.out) + plane + ((size_t)oh * a.ow + ow) * px + 4 * g));
      }
    } else {
      uint8_t *block = static_cast<uint8_t *>(a.out) + plane;
      unsigned pk[PX], old[PX];
#pragma unroll
      for (int e = 0; e < PX; ++e) pk[e] = old[e] = 0u;
      if (a.with_sum)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) load_old_row<A>(old + M * i, block, r0 + i, g, th, tw, a.oh, a.ow, px);
      auto quantize = [&](auto out_c, auto relu_c, auto sum_c) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          pack_channel<decltype(out_c)::value, A, PX>(y[k], comp_of(bias, k), k, decltype(relu_c)::value, a.out_repS, a.out_z,
                                                      decltype(sum_c)::value, old, pk);
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
      for (int i = 0; i < ROWS; ++i) store_row<A>(pk + M * i, block, r0 + i, g, valid, th, tw, a.oh, a.ow, px);
    }
  }
}

// The workgroups of form 0, 1, 2 = 16 channels x 16 tiles, 32 x 16, 32 x 32 for so many blocks of 16 tiles and of 16 channels, and which of them an
// XCD takes: a rectangle of nxx x nyy, the one of least reading (its share of the weights and its share of the tiles) among those that give each
// of its 32 CUs one workgroup at most, if there are any.
struct ColsGrid {
  int nx, ny;     // groups of tiles, of channels
  int slots;      // log2 of the XCDs beside each other along the tiles
  int nxx, nyy;
};
static ColsGrid cols_grid(int blocks, int oc2, int form)
{
  const int ro = form >= 1 ? 2 : 1, rt = form == 2 ? 2 : 1;
  ColsGrid g;
  g.nx = (blocks + rt - 1) / rt;
  g.ny = (oc2 + ro - 1) / ro;
  long long best = -1;
  bool best_fits = false;
  for (int xa = 0; xa <= 3; ++xa) {
    const int nxx = (g.nx + (1 << xa) - 1) >> xa, nyy = (g.ny + (8 >> xa) - 1) / (8 >> xa);
    const long long read = (long long)nxx * rt + (long long)nyy * ro;   // (times A * A * ic2 * 256 bytes)
    const bool fits = (long long)nxx * nyy <= 32;
    if (best >= 0 && (fits == best_fits ? read >= best : best_fits)) continue;
    best = read;
    best_fits = fits;
    g.slots = xa;
    g.nxx = nxx;
    g.nyy = nyy;
  }
  return g;
}
static bool cols_one_round(int blocks, int oc2, int form)
{
  const ColsGrid g = cols_grid(blocks, oc2, form);
  return (long long)g.nxx * g.nyy <= 32;
}

// The form for a layer: 0, 1, 2 = 16 channels x 16 tiles, 32 x 16, 32 x 32 a workgroup, -1 = none.  Each is the fastest while every
// workgroup has a CU of its own, the smaller one first; a second round costs as much as the first, and the other kernels share what
// they read among more products.  Fused stage, other tensors on every call, us: the kernel that ran before / the three forms, at
// so many workgroups of 16 x 16 (16 x 16 against the channels shared out among the waves, a form that is gone, resident weights
// or the ring):
//   tile size 6: 64 channels 7.9 / 6.4 7.9 8.9 (256), 9.0 / 9.6 8.4 9.0 (512), 9.0 / - 14.3 9.5 (1024); 128 channels 9.9 / 7.2 8.1 10.4 (256),
//     11.0 / 10.5 8.6 10.5 (512), 11.0 / - 15.3 11.1 (1024); 256 channels 10.7 / 8.9 10.2 12.6 (256), 15.7 / 14.7 10.8 13.0 (512), 17.7 / - 19.4 14.0 (1024), 21.7 / - - 23.4
//     (1280); 512 channels 15.7 / 12.6 14.2 18.1 (256), 21.7 / 22.5 15.3 18.3 (512), 22.9 / - 28.1 20.0 (1024), 28.8 / - - 34.4 (1280); 1024 channels 39.9 / 24.1 22.7
//     28.9 (256), 43.0 / 45.5 26.5 29.9 (512), 50.6 / - 48.5 32.2 (1024)
//   tile size 5: 64 channels 6.2 / 5.0 6.7 7.3 (256), 5.8 / 6.9 7.9 7.7 (320); 128 channels 8.2 / 6.4 7.7 8.5 (256), 8.5 / 8.1 7.5 8.9 (512), 9.0 / - 12.2 9.2 (1024);
//     256 channels 8.6 / 7.2 8.4 10.4 (256), 11.9 / 10.6 8.6 10.6 (512), 12.4 / - 15.4 11.3 (1024); 512 channels 17.1 / - 21.3 16.0 (1024)
//   tile size 4: 128 channels 5.0 / 5.6 4.8 6.0 (256), 6.3 / 7.4 5.4 6.2 (512); 256 channels 6.9 / 5.9 6.2 7.4 (256), 7.7 / 8.4 6.3 7.4 (512), 7.9 / - 8.2 7.5 (640);
//     512 channels 9.0 / 7.9 8.0 9.7 (256), 11.5 / - 12.9 10.7 (1024)
// An XCD has 32 of the CUs, and takes a rectangle of the workgroups: 49 x 5 of them do not come to one round on any XCD (at best 35
// on one), and cost two.  Then the next form is the faster one, or none: 160 -> 160, 49 blocks of tiles, tile size 6, with the input transform
// 16.6 / 21.1 with 32 x 16; 453 -> 275, 54 blocks, tile size 5 28.9 / 36.5 with 32 x 32; 184 -> 80, 49 blocks 16.7 with 16 x 16, 15.2 with 32 x 16.
// A few workgroups gain as much as a chip full of them: 288 / 512 -> 16 to 256, one image of 7 x 7 or 14 x 14, with the input transform, tile size 6 19.2 to
// 23.5 us (ring) / 11.7 to 13.2 (16 x 16), 5 14.3 to 19.2 / 9.9 to 11.5, 4 10.7 to 13.0 / 8.6 to 9.5.
// 32 x 32 with up to 256 input channels only from 192 output channels on: with fewer, the layer has so many tiles that they are what
// it reads, and resident weights read them once (with the input transform, 256 -> 64, 160 blocks of tiles 28.7 / 29.7; 192 -> 32, 390
// blocks 34.3 / 36.5).
int wino_cols_pick(const WinoFusedArgs &a)
{
  const int A = a.tile ? a.tile : 6, nks = (a.ic2 + 3) / 4, blocks = (a.t + 15) / 16;
  if (a.units_pad < 4 * nks || (a.out_type == EHIP_F32 && a.with_sum)) return -1;
  if ((long long)A * A * a.units_pad * a.ocpp * 16 > 0x7fffffffll || (long long)((a.t + 31) / 32) * A * A * a.ic2 * 512 > 0x7fffffffll) return -1;
  if (const char *env = getenv("EHIP_WINO_COLS")) return env[0] >= '0' && env[0] <= '2' ? env[0] - '0' : -1;
  // (a switch that asks for one of the other forms)
  for (const char *k : {"EHIP_WINO_LANES", "EHIP_WINO_LANES_WRES", "EHIP_WINO_LANES_SLOTS", "EHIP_WINO_LANES_WAVES", "EHIP_WINO_RING"})
    if (getenv(k)) return -1;
  if (cols_one_round(blocks, a.oc2, 0)) return A == 4 && nks < 3 ? -1 : 0;
  if (cols_one_round(blocks, a.oc2, 1)) return A == 6 || nks >= 2 ? 1 : -1;
  if (cols_one_round(blocks, a.oc2, 2)) return nks > 4 || (nks >= (A == 4 ? 4 : 3) && a.oc2 >= 12) ? 2 : -1;
  return -1;
}

hipError_t plan_wino_gemm_output_cols(LaunchPlan &plan, const WinoFusedArgs &a0, int form)
{
  WinoFusedArgs a = a0;
  const int A = a.tile ? a.tile : 6;
  const int ro = form >= 1 ? 2 : 1, blocks = form == 2 ? 2 : 1;
  void (*kernel)(const WinoFusedArgs *, void *, const float *) = nullptr;
#define EHIP_WC(A) kernel = form == 0 ? k_wino_gemm_output_lanes_cols<A, 1, 1> : (form == 1 ? k_wino_gemm_output_lanes_cols<A, 2, 1> : k_wino_gemm_output_lanes_cols<A, 2, 2>)
  if (A == 4) EHIP_WC(4);
  else if (A == 5) EHIP_WC(5);
  else EHIP_WC(6);
#undef EHIP_WC
  const ColsGrid g = cols_grid((a.t + 15) / 16, a.oc2, form);
  a.nx = g.nx; a.ny = g.ny; a.slots = g.slots;
  const dim3 grid(8 * g.nxx, g.nyy);
  const size_t lds = (size_t)ro * blocks * (A == 4 ? A : A - 2) * A * 1024 + (size_t)A * 3 * A * 64 * ro;
  static const char *const names[] = {"k_wino_gemm_output_lanes_cols<16,16>", "k_wino_gemm_output_lanes_cols<32,16>",
                                      "k_wino_gemm_output_lanes_cols<32,32>"};   // channels, tiles of a workgroup
  plan.name = names[form];
  return plan_set(plan, kernel, grid, dim3(64 * A), lds, a, ArgBlock{}, ArgOut{a.out}, ArgBias{});
}

}  // namespace ehip
