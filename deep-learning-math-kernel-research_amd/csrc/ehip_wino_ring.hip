// Choice and launch of the ring kernels (ehip_wino_ring.hpp).
#include "ehip_internal.hpp"

namespace ehip {

namespace {
// Workgroups of oct channels x tt tiles: the channel blocks, the blocks of tiles, the workgroups per XCD and channel block
// with per_cu of them on a CU, and how many blocks the longest walk of a workgroup takes
struct RingGrid {
  int ny, nx, slots, rounds;
  int workgroups() const { return 8 * ny * slots; }
};
RingGrid ring_grid(const WinoFusedArgs &a, int oct, int tt, int per_cu)
{
  RingGrid g;
  g.ny = (a.oc2 * 16 + oct - 1) / oct;
  g.nx = (a.t + tt - 1) / tt;
  g.slots = 32 * per_cu / g.ny;
  const int need = (g.nx + 7) / 8;
  g.slots = g.slots < 1 ? 1 : (g.slots < need ? g.slots : need);
  g.rounds = (g.nx + 8 * g.slots - 1) / (8 * g.slots);
  return g;
}
}  // namespace

// the form for a layer (ring_form), -1 = not one for these kernels
int wino_ring_pick(const WinoFusedArgs &a)
{
  const int A = a.tile ? a.tile : 6;
  const int nks64 = (a.ic2 + 3) / 4;
  // whole stages of k-steps; 32-bit offsets into the weights
  const int kc = nks64 <= 4 ? 4 : (nks64 <= 6 ? 6 : (nks64 + 1) / 2 * 2);
  if (a.units_pad < 4 * kc || (a.out_type == EHIP_F32 && a.with_sum)) return -1;
  if ((long long)A * A * a.units_pad * a.ocpp * 16 > 0xffffffffll) return -1;
  for (const char *other : {"EHIP_WINO_LANES", "EHIP_WINO_LANES_WRES"})   // (the other forms asked for)
    if (const char *env = getenv(other)) if (env[0] == '0') return -1;
  if (const char *env = getenv("EHIP_WINO_RING")) {   // (0, 1, 2: that form where it exists; anything else: none)
    const int form = env[0] - '0';
    return form == 2 ? (nks64 == 4 ? 2 : -1) : (form >= 0 && form < 2 && nks64 > 4 ? form : -1);
  }
  // 193-256 channels: from three quarters of a workgroup per CU (N = 16, 256 -> 256: at 28 x 28 with tile size 5, 200
  // workgroups, 28.0 -> 25.1 us a layer; with tile size 6, 104, 23.3 with resident weights and 28.7 here; 56 x 56 at
  // N = 64, 1568, 131 -> 120).  Fewer channels: the resident weights' form stays (192 -> 192 at 28 x 28: 18.6 / 19.5).
  if (nks64 <= 4) {
    const RingGrid g = ring_grid(a, 32, 64, 2);
    return nks64 == 4 && (long long)g.nx * g.ny >= 192 ? 2 : -1;
  }
  // More: the longest walk of a workgroup (times the rounds of workgroups, with more channel blocks than the chip takes at
  // once) times what a block costs: 36 with large blocks, with small ones 20 alone on a CU and 30 with two.  That is the
  // time in us with 512 channels and tile size 6; with other channel counts (272 to 2048) and tile sizes all three move
  // together.  Fused stage, us, 64 x 64 / 32 x 32 / the general kernel, u8 in and s8 out:
  //   512 -> 256, tiles of 14 x 14 images: N = 1 31 / 19 / 23, N = 64 35 / 21 / 25, N = 96 35 / 27 / 47, N = 128 36 / 30 / 35,
  //   N = 192 36 / 43 / 65, N = 256 40 / 58 / 70;  288 -> 320 at 28 x 28, N = 32 (a second round for few blocks) 29 / 34 / 54
  // 565 layers of 16 to 1500 output channels, 1 to 64 images and every tile size: two of them 5 and 10 % behind the best.
  const RingGrid large = ring_grid(a, 64, 64, 1), small = ring_grid(a, 32, 32, 2);
  const int large_cost = 36 * large.rounds * ((large.workgroups() + 255) / 256);
  const int small_cost = (small.workgroups() <= 256 ? 20 : 30) * small.rounds * ((small.workgroups() + 511) / 512);
  const int form = large_cost < small_cost ? 0 : 1;
  // More than 512 channels (a position's stages in a loop, the requests worked out at run time: a small block's ten k-steps
  // take 32 us where eight in straight-line code take 20) and no more workgroups of the general kernel than CUs: that one, with tile size 6 always, with 5 where small
  // blocks would share a CU or for up to 64 output channels.  1024 -> 256, tile size 6: 16 tiles 74 / 46 / 38, 1024 tiles
  // 75 / 48 / 41, 1536 (two rounds there) 75 / 66 / 78, 2048 76 / 68 / 53, 3072 76 / 94 / 99; tile size 5: 25 tiles
  // 51 / 33 / 34, 1600 52 / 49 / 41; 640 -> 64, 50 tiles 36 / 24 / 18; tile size 4: 20 / 30 small / general, always a ring.
  if (nks64 > 8 && A >= 5 && wino_general_workgroups(a, nullptr) <= 256 &&
      (A == 6 || a.oc2 <= 4 || (form == 1 && small.workgroups() > 256)))
    return -1;
  return form;
}

hipError_t plan_wino_gemm_output_ring(LaunchPlan &plan, const WinoFusedArgs &a0, int form)
{
  WinoFusedArgs a = a0;
  const int A = a.tile ? a.tile : 6, AA = A * A;
  const int nks64 = (a.ic2 + 3) / 4;
  const RingForm f = A == 4 ? wino_ring_form4(form, nks64) : (A == 5 ? wino_ring_form5(form, nks64) : wino_ring_form6(form, nks64));
  const size_t lds = (size_t)f.stage_kb * 1024 * f.stages + (size_t)AA * 3 * f.oct * 4;
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  a.nkc = (nks64 + f.kc - 1) / f.kc;
  int per_cu = (int)(160 * 1024 / lds);
  if (per_cu > 8 / f.waves) per_cu = 8 / f.waves;
  const RingGrid g = ring_grid(a, f.oct, f.tt, per_cu);
  a.nx = g.nx; a.ny = g.ny; a.slots = g.slots;
  static const char *const names[] = {"k_wino_gemm_output_lanes_ring<64,64>", "k_wino_gemm_output_lanes_ring<32,32>",
                                      "k_wino_gemm_output_lanes_ring<32,64>"};   // channels, tiles of a workgroup
  plan.name = names[form];
  return plan_set(plan, f.kernel, dim3(g.workgroups()), dim3(64 * f.waves), lds, a, ArgBlock{}, ArgOut{a.out}, ArgBias{});
}

}  // namespace ehip
