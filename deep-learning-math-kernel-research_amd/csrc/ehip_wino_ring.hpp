// Winograd GEMMs + output transform with BOTH operands streamed through an LDS ring: the form for layers whose operand
// stream is what bounds the fused stage (more than 256 input channels; 256 with many tiles).
//
// Replaces, for those layers, elx_int8_conv_wino_gemm_t::execute + trans_output as the reference's fused schedule
// runs them per thread (a161, src/elx_int8_conv_wino_xopt.hpp:21-179; src/elx_int8_conv_wino_gemm.cpp:23-205,
// src/elx_conv_wino_trans_output.cpp:212-423).
//
// What bounds it: a CU takes 48 bytes a clock from its L2 while all of them do (56 where the L1 has them), so the product of a weight and a tile byte is only as cheap
// as the block of channels x tiles they are shared in.  With the weights of 16 channels resident (ehip_wino_lanes.hip) a
// byte of the transformed input feeds 16 products; a workgroup of 64 channels x 64 tiles makes it 32 for both operands, and
// keeps no more than 16 + 4 running values per output channel and tile in a lane (Fold) instead of all 36 positions,
// because the positions are finished one after the other: a position's 64 x 64 sums are requantized and folded into the
// output transform while the next position is multiplied.
// That still takes all of the 256 registers that a wave has with two on a SIMD: at tile size 6 the forms of 64 tiles (0 and
// 2) keep 11 to 15 values in scratch memory, stored ahead of the loop over the positions and reloaded in the output phase
// (2 MB of writes beside 51 MB of output, 256 -> 256 at 56 x 56, N = 64).  A reload waits by the counter that the requests for
// the next block of tiles are in as well, so it waits for those, too.
// The operands travel global memory -> LDS without registers, five stages ahead, and LDS -> registers one stage ahead; one
// barrier per stage.  512 -> 512 at 28 x 28, N = 64 (u8 in, s8 out): 114-117 us with the weights resident in two passes over
// half of the columns each (a form that is gone), 69-74 us here, of which the L1 stream is 40 us and the vector work of the
// transforms, which only partly hides behind it, 25; 256 -> 256 at 56 x 56 90 -> 78 us, f32 in and out 122 -> 100 us.
// A workgroup walks whole blocks of 64 tiles: where their number does not divide over the workgroups of a channel block, the
// last round is short (256 -> 256 at 56 x 56, N = 64: 196 blocks over 64 columns of workgroups, four rounds for 3.06).
// Tried: splitting the channels over the waves 2 x 4 instead of 4 x 2 (twice the reads of per-channel constants: 4 %
// slower); all positions unrolled (60 to 120 KB of instructions: 0.28 us per KB and block of tiles); the two waves of a SIMD
// folding in different stages (the running values are copied where the branches meet: 10 % slower); four k-steps per
// stage (the ring is then four stages deep and starves).
//
// Compiled with the accumulators in the ordinary vector registers, like ehip_wino_lanes.hip.
#ifndef EHIP_WINO_RING_HPP
#define EHIP_WINO_RING_HPP
#include "ehip_wino_fold.hpp"
#include "ehip_wino_pack.hpp"

namespace ehip {

namespace {

// 16 bytes per lane from global memory straight into LDS (lane i's piece lands at lds_addr + 16 i); assembly the
// compiler does not track, so that its own waits never cover these loads: the kernel waits by count.
__device__ __forceinline__ void dma16(const void *sbase, unsigned voff, unsigned lds_addr)
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "m0");
#else
  (void)sbase;
  (void)voff;
  (void)lds_addr;
#endif
}
// at most N of the wave's vector-memory operations still in flight; then the barrier.  (Nothing waits for the wave's LDS
// reads here: a slot is requested again only two barriers after its operands were read, one after they were multiplied.)
template <int N>
__device__ __forceinline__ void wait_and_barrier()
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory");
#endif
}
__device__ __forceinline__ void wait_all_loads()
{
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#endif
}

// position visited i-th: runtime form, for the cursor of the loads
template <int A>
__device__ __forceinline__ int position_at(int i)
{
  const int ci = i / A, ri = i - A * ci;
  return A * Fold<A>::order(ri) + Fold<A>::order(ci);
}

}  // namespace

// Workgroup = OCT output channels x TT tiles at all positions, WO x WT waves of 16 RO channels x 16 RT tiles each.
// A stage of the ring holds KC k-steps of 64 channels of ONE position of both operands (NKC stages per position; 0: a.nkc of
// them); the R stages run on over positions and over the blocks of tiles that the workgroup walks.
template <int A, int RO, int RT, int WO, int WT, int KC, int NKC, int R>
__global__ __launch_bounds__(64 * WO * WT, 2) void k_wino_gemm_output_lanes_ring(const WinoFusedArgs *rest, void *out, const float *bias_)
{
  WinoFusedArgs a = load_args(rest);
  a.out = out; a.bias = bias_;
  constexpr int NWV = WO * WT, TB = 64 * NWV;
  constexpr int OCT = 16 * RO * WO, TT = 16 * RT * WT;
  constexpr int AA = A * A, M = A - 2;
  constexpr int NA = OCT * KC / 16, NB = TT * KC / 16;        // loads of 1 KB per stage
  constexpr int LPW = (NA + NB + NWV - 1) / NWV;              // per wave
  constexpr int STAGE = (NA + NB) * 1024, RING = R * STAGE;
  constexpr int FLIGHT = (R - 3) * LPW;
  constexpr bool DUP = (NA + NB) % NWV != 0;                  // some waves load the last piece once more
  extern __shared__ float4 lds[];
  constexpr int CL = RING / 16;                               // constants behind the ring: [AA][3][OCT / 4 quads]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wo = wave % WO, wt = wave / WO;
  const int l16 = lane & 15, g = lane >> 4;
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int by = seq % a.ny;
  const int item_step = 8 * a.slots;
  const int item0 = (seq / a.ny) * 8 + xcd;
  if (item0 >= a.nx) return;          // whole workgroup
  const int oc0 = by * OCT;
  const int oc_real = a.oc2 * 16;
  const int nblk = (a.t + 31) >> 5;
  const int nkc = NKC ? NKC : a.nkc;
  // ---- loads: the wave's LPW pieces of a stage ---------------------------------------------------------------
  // piece j of a stage: j < NA weights (LDS [unit][OCT rows]: row 16 b + r of the stage = MFMA row r of channel block b,
  // taken from its place in the packed group of 32), else tiles (LDS [unit][TT tiles])
  unsigned voff[LPW], vrow[LPW];
  bool is_a[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    int j = wave + NWV * i;
    j = j < NA + NB ? j : NA + NB - 1;
    is_a[i] = j < NA;
    if (is_a[i]) {
      const int c = j * 64 + lane, unit = c / OCT, s = c % OCT, s32 = s & 31;
      const int row = (s & ~31) + 8 * ((s32 & 15) >> 2) + 4 * (s32 >> 4) + (s32 & 3);
      voff[i] = (unsigned)(unit * a.ocpp + row) * 16u;
      vrow[i] = 0;
    } else {
      const int c = (j - NA) * 64 + lane, unit = c / TT, tile = c % TT;
      voff[i] = (unsigned)(unit * 512 + (tile & 31) * 16);
      vrow[i] = (unsigned)(tile >> 5);
    }
  }
  const unsigned w_pos = (unsigned)a.units_pad * (unsigned)a.ocpp * 16u, w_kc = (unsigned)a.ocpp * (64u * KC);   // bytes (the launcher
  const unsigned t_pos = (unsigned)a.ic2 * 512u, t_kc = 2048u * KC;                                              // checks 32 bits)
  const unsigned long long t_blk = (unsigned long long)AA * t_pos;
  const uint8_t *w0 = reinterpret_cast<const uint8_t *>(a.w) + (size_t)oc0 * 16;
  const uint8_t *pf_base;             // the tiles that the requests are in
  unsigned voff_b[LPW];
  auto enter = [&](int item) {
    const int b32 = TT >= 32 ? item * (TT / 32) : item * TT / 32;
    pf_base = a.tin + b32 * t_blk + (TT < 32 ? (item * TT & 31) * 16 : 0);
#pragma unroll
    for (int i = 0; i < LPW; ++i)   // (a block past the last one reads the item's first)
      voff_b[i] = voff[i] + (TT > 32 && b32 + (int)vrow[i] < nblk ? vrow[i] * (unsigned)t_blk : 0u);
  };
  unsigned pf_lds = wave * 1024;      // where the next stage's first piece goes
  auto request = [&](int p, int kc) {
    const uint8_t *pa = w0 + ((unsigned)p * w_pos + (unsigned)kc * w_kc);
    const uint8_t *pb = pf_base + ((unsigned)p * t_pos + (unsigned)kc * t_kc);
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      unsigned dst = pf_lds + NWV * 1024 * i;
      if (DUP && i == LPW - 1 && wave + NWV * i >= NA + NB) dst = pf_lds - wave * 1024 + (NA + NB - 1) * 1024;   // same bytes
      dma16(is_a[i] ? pa : pb, voff_b[i], dst);
    }
    pf_lds += STAGE;
    if (pf_lds >= RING) pf_lds -= RING;
  };
  // The order of the stages: column by column of the positions, rows inside, each in Fold's order.  With NKC > 0 a column's
  // stages are straight-line code and the request that a stage makes lies R - 1 stages on: its row and k-steps are known,
  // its column is ci + a known number.
  constexpr int NK = NKC ? NKC : 1, SC = A * NK;   // stages of a column
  int rq_pos = 0, rq_kc = 0;          // (NKC = 0: the cursor of the requests)
  int pf_item = item0;
  auto pf_next_item = [&]() {         // (behind the last block: its head again, unused)
    if (pf_item + item_step < a.nx) pf_item += item_step;
    enter(pf_item);
  };
  auto row_order = [](int i) { return (int)Fold<A>::kOrder[i]; };
  auto request_at = [&](int ci, int q) {   // NKC > 0: the q-th stage behind the start of column ci, q may lie in the next columns
    const int dc = q / SC, qq = q % SC;
    if (qq == 0 && ci + dc == A) pf_next_item();
    request(A * row_order(qq / NK) + Fold<A>::order(ci + dc), qq % NK);
  };
  auto request_next = [&]() {         // NKC = 0
    request(position_at<A>(rq_pos), rq_kc);
    if (++rq_kc == nkc) {
      rq_kc = 0;
      if (++rq_pos == AA) {
        rq_pos = 0;
        pf_next_item();
      }
    }
  };
  enter(item0);
#pragma unroll
  for (int s = 0; s < R - 1; ++s) {
    if (NKC) request_at(0, s);
    else request_next();
  }
  // ---- constants ---------------------------------------------------------------------------------------------
  {
    constexpr int Q = OCT / 4, NCELL = AA * 3 * Q;
    for (int idx = tid; idx < NCELL; idx += TB) {
      const int p = idx / (3 * Q), rem = idx - 3 * Q * p, arr = rem / Q, q = rem % Q;
      const float *src = a.scale + (size_t)arr * AA * a.ocpp;   // (scale, shift, compensation: one allocation, [3][AA][ocpp])
      lds[CL + idx] = *reinterpret_cast<const float4 *>(src + (long long)p * a.ocpp + oc0 + 4 * q);
    }
  }
  const int px = a.out_nhwc ? a.oc2 * 16 : 16;
  // the lane's cells: 16-byte cells from the start of the LDS; opaque, so that reads are base + immediate offset
  const int la = g * OCT + RO * wo * 16 + l16, lb = NA * 64 + g * TT + RT * wt * 16 + l16;
  int lc = CL + RO * wo * 4 + g;
  asm volatile("" : "+v"(lc));
  int ring = 0;                       // cells from the start of the ring to the stage being multiplied
  v4i va[KC][RO], vb[KC][RT];         // operands, one stage ahead of the matrix instructions
  auto read = [&](int ring_at, int ks) {
    const v4i *l = reinterpret_cast<const v4i *>(lds) + ring_at;
#pragma unroll
    for (int j = 0; j < RT; ++j) vb[ks][j] = l[lb + ks * 4 * TT + 16 * j];
#pragma unroll
    for (int b = 0; b < RO; ++b) va[ks][b] = l[la + ks * 4 * OCT + 16 * b];
  };
  auto next_of = [&](int r) { return r + STAGE / 16 == RING / 16 ? 0 : r + STAGE / 16; };
  __syncthreads();                    // the constants are in LDS
  wait_and_barrier<(R - 2) * LPW>();  // the first stage has landed
#pragma unroll
  for (int ks = 0; ks < KC; ++ks) read(0, ks);

  for (int item = item0; item < a.nx; item += item_step) {
    float Y[RO * RT][4][M][4];            // [block][channel][row][running values of the second dimension]
    float C[RO * RT][4][4];               // [block][channel][running values of the first dimension]
    float P[A == 4 ? AA : 1][RO * RT][4]; // tile size 4: the requantized positions
    v4i acc[2][RO * RT];
    float4 sc[RO], sh[RO];                // of the position in acc[]
    // Requantization and folding of a column's ri-th position.  They run one position late, between the matrix instructions
    // of the next one.
    auto finish = [&](int ci, int ri) {
#pragma unroll
      for (int b = 0; b < RO; ++b) {
        const float scv[4] = {sc[b].x, sc[b].y, sc[b].z, sc[b].w}, shv[4] = {sh[b].x, sh[b].y, sh[b].z, sh[b].w};
#pragma unroll
        for (int j = 0; j < RT; ++j) {
          const int e = b * RT + j;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float x = __builtin_fmaf((float)acc[ri & 1][e][k], scv[k], shv[k]);
            if constexpr (A == 4) {
              P[A * ri + ci][e][k] = x;
              asm volatile("" : "+v"(P[A * ri + ci][e][k]));
            } else {
              fold_step<A>(ri, C[e][k], x, std::make_integer_sequence<int, A>{});
              pin(C[e][k], ri);   // (left to itself the compiler defers the folding and keeps every requantized value instead)
            }
          }
        }
      }
    };
    auto column = [&](int ci) {
      const int lcol = lc + Fold<A>::order(ci) * (3 * (OCT / 4));
#pragma unroll
      for (int ri = 0; ri < A; ++ri) {
        const int lp = lcol + A * row_order(ri) * (3 * (OCT / 4));
        auto stage = [&](int kc, bool first) {
          wait_and_barrier<FLIGHT>();   // the stage behind this one has landed, and everyone has left the one before it
          const int ring_n = next_of(ring);
          if (first) {
            // (the accumulators start from the compensation 128 * sum(weights) of their (position, channel))
#pragma unroll
            for (int b = 0; b < RO; ++b) {
              const float4 cf = lds[lp + 2 * (OCT / 4) + 4 * b];
#pragma unroll
              for (int j = 0; j < RT; ++j)
                acc[ri & 1][b * RT + j] = v4i{__float_as_int(cf.x), __float_as_int(cf.y), __float_as_int(cf.z), __float_as_int(cf.w)};
            }
          }
#pragma unroll
          for (int ks = 0; ks < KC; ++ks) {
#pragma unroll
            for (int j = 0; j < RT; ++j)
#pragma unroll
              for (int b = 0; b < RO; ++b)
                acc[ri & 1][b * RT + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(va[ks][b], vb[ks][j], acc[ri & 1][b * RT + j], 0, 0, 0);
            read(ring_n, ks);
            // (the requests behind the first matrix instructions: a request waits its turn at the memory pipe, and everything
            // behind it in the wave's order waits too)
            if (ks == 0) {
              if (NKC) request_at(ci, ri * NK + kc + R - 1);
              else request_next();
            }
            if (first && ks == 0) {
              if (ri > 0) finish(ci, ri - 1);
#pragma unroll
              for (int b = 0; b < RO; ++b) {
                sc[b] = lds[lp + 4 * b];
                sh[b] = lds[lp + (OCT / 4) + 4 * b];
              }
            }
          }
          ring = ring_n;
          __builtin_amdgcn_sched_barrier(0);
        };
        stage(0, true);
        if (NKC) {
#pragma unroll
          for (int kc = 1; kc < NKC; ++kc) stage(kc, false);
        } else {
          for (int kc = 1; kc < nkc; ++kc) stage(kc, false);
        }
      }
      finish(ci, A - 1);
    };
    if constexpr (A == 4) {
#pragma unroll
      for (int ci = 0; ci < A; ++ci) column(ci);
    } else {
      // A loop over the columns: unrolled, the A x A positions are 50 to 120 KB of instructions, more than the instruction
      // cache holds, and every block of tiles waits for them (0.28 us a KB).  What differs from column to column is the
      // second fold: separate blocks, each with an opaque statement inside, or they become selects between all of them.
#pragma unroll
      for (int e = 0; e < RO * RT; ++e)
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int r = 0; r < M; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) Y[e][k][r][q] = 0.0f;
#pragma unroll 1
      for (int ci = 0; ci < A; ++ci) {
        column(ci);
        auto fold_rows = [&](auto kc_) {
          constexpr int K = decltype(kc_)::value;
          int c = ci;
          asm volatile("" : "+s"(c));   // (every test stands alone)
          if (c == K) {
#pragma unroll
            for (int e = 0; e < RO * RT; ++e)
#pragma unroll
              for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < M; ++r) Fold<A>::template step_in_place<K>(Y[e][k][r], Fold<A>::result(C[e][k], r));
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
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const int t = item * TT + (RT * wt + j) * 16 + l16;
      const int tt = t < a.t ? t : 0;
      const int n = tt / a.nt;
      const int rem = tt - n * a.nt;
      const int th = rem / a.wt;
      const int tw = rem - th * a.wt;
#pragma unroll
      for (int b = 0; b < RO; ++b) {
        const int e = b * RT + j;
        const int oc = oc0 + (RO * wo + b) * 16 + 4 * g;
        const bool valid = t < a.t && oc < oc_real;
        // (lanes without a tile or channel of their own take part with tile 0 / channel 0 and store nothing)
        const int occ = oc < oc_real ? oc : 0;
        float4 bias = make_float4(0.f, 0.f, 0.f, 0.f);
        if (a.with_bias) bias = *reinterpret_cast<const float4 *>(a.bias + occ);
        const size_t plane = a.out_nhwc ? (size_t)n * a.oh * a.ow * a.oc2 * 16 + (occ >> 4) * 16
                                        : ((size_t)n * a.oc2 + (occ >> 4)) * a.oh * a.ow * 16;
        auto value = [&](int k, float *y) {
          if constexpr (A == 4) {
            float f[AA];
#pragma unroll
            for (int q = 0; q < AA; ++q) f[q] = P[q][e][k];
            wino::tile_output<4>(f, y);
          } else {
#pragma unroll
            for (int r = 0; r < M; ++r)
#pragma unroll
              for (int c = 0; c < M; ++c) y[M * r + c] = Fold<A>::result(Y[e][k][r], c);
          }
        };
        if (a.out_type == EHIP_F32) {
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
          auto quantize = [&](auto out_c, auto relu_c, auto sum_c) {
            constexpr int OUT = decltype(out_c)::value;
            constexpr bool RELU = decltype(relu_c)::value, SUM = decltype(sum_c)::value;
            if (SUM) load_old_cells<A>(old, block, g, th, tw, a.oh, a.ow, px);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              float y[M * M];
              value(k, y);
              pack_channel<OUT, A, (A - 2) * (A - 2), true>(y, comp_of(bias, k), k, RELU, a.out_repS, a.out_z, SUM, old, pk);
#pragma unroll
              for (int q = 0; q < M * M; ++q) asm volatile("" : "+v"(pk[q]));
              __builtin_amdgcn_sched_barrier(0);
            }
          };
          using U8C = std::integral_constant<int, EHIP_U8>;
          using S8C = std::integral_constant<int, EHIP_S8>;
          auto relu_sum = [&](auto out_c) {
            if (a.with_sum) {
              if (a.with_relu) quantize(out_c, std::true_type{}, std::true_type{});
              else quantize(out_c, std::false_type{}, std::true_type{});
            } else {
              if (a.with_relu) quantize(out_c, std::true_type{}, std::false_type{});
              else quantize(out_c, std::false_type{}, std::false_type{});
            }
          };
          if (a.out_type == EHIP_U8) relu_sum(U8C{});
          else relu_sum(S8C{});
          store_cells<A>(pk, block, g, valid, th, tw, a.oh, a.ow, px);
        }
      }
    }
  }
  wait_all_loads();   // (the requests behind the last stage still write this workgroup's LDS)
}

// Form 0: 64 channels x 64 tiles, eight waves, one workgroup per CU.  A stage of two k-steps (16 KB) takes the L1 340
// clocks at 48 bytes a clock, the matrix cores 134 and the LDS less than the L1 (203 clocks of reads beside
// the 16 KB coming in).  Form 1: 32 x 32, four waves, two workgroups per CU: twice the operand bytes per product, for
// layers of few tiles.  Form 2: 32 x 64, four waves, two workgroups per CU that hide each other's transforms and stores,
// which with 256 input channels weigh more than the operand stream.
template <int A>
RingForm ring_form(int form, int nks)
{
#define EHIP_RING(RT, WO, WT, KC, NKC, R) \
  RingForm{k_wino_gemm_output_lanes_ring<A, 1, RT, WO, WT, KC, NKC, R>, 16 * WO, 16 * RT * WT, WO * WT, (WO + RT * WT) * KC, R, KC}
  if (form == 2) return EHIP_RING(2, 2, 2, 2, 2, 5);
  if (form == 0) {
    if (nks <= 6) return EHIP_RING(2, 4, 2, 3, 2, 5);
    if (nks <= 8) return EHIP_RING(2, 4, 2, 2, 4, 8);
    return EHIP_RING(2, 4, 2, 2, 0, 8);
  }
  if (nks <= 6) return EHIP_RING(1, 2, 2, 3, 2, 5);
  if (nks <= 8) return EHIP_RING(1, 2, 2, 2, 4, 7);
  return EHIP_RING(1, 2, 2, 2, 0, 7);
#undef EHIP_RING
}

}  // namespace ehip
#endif
