// Choice and launch of the ring kernels (ehip_wino_ring.hpp).
#include "ehip_internal.hpp"

namespace ehip {

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
  auto items = [&](int oct, int tt) { return (long long)((a.t + tt - 1) / tt) * ((a.oc2 * 16 + oct - 1) / oct); };
  if (const char *env = getenv("EHIP_WINO_RING")) {   // (0, 1, 2: that form where it exists; anything else: none)
    const int form = env[0] - '0';
    return form == 2 ? (nks64 == 4 ? 2 : -1) : (form >= 0 && form < 2 && nks64 > 4 ? form : -1);
  }
  // 193-256 channels: from three quarters of a workgroup per CU (N = 16, 256 -> 256: at 28 x 28 with tile size 5, 200
  // workgroups, 28.0 -> 25.1 us a layer; with tile size 6, 104, 23.3 with resident weights and 28.7 here; 56 x 56 at
  // N = 64, 1568, 131 -> 120).  Fewer channels: the resident weights' form stays (192 -> 192 at 28 x 28: 18.6 / 19.5).
  if (nks64 <= 4) return nks64 == 4 && items(32, 64) >= 192 ? 2 : -1;
  // More: rounds of workgroups over the chip times what a round takes with 512 channels (36 us; small blocks 20 us alone on
  // a CU, 30 us with two).  N = 64, 512 -> 512: 28 x 28 99 (large) / 124 us (small) a layer, 14 x 14 49 / 44, 7 x 7 41 / 28.
  const long long large = items(64, 64), small = items(32, 32);
  return 36 * ((large + 255) / 256) < (small <= 256 ? 20 : 30) * ((small + 511) / 512) ? 0 : 1;
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
  a.nx = (a.t + f.tt - 1) / f.tt;
  a.ny = (a.oc2 * 16 + f.oct - 1) / f.oct;
  int per_cu = (int)(160 * 1024 / lds);
  if (per_cu > 8 / f.waves) per_cu = 8 / f.waves;
  int slots = 32 * per_cu / a.ny;
  slots = slots < 1 ? 1 : slots;
  const int need = (a.nx + 7) / 8;
  a.slots = slots < need ? slots : need;
  static const char *const names[] = {"k_wino_gemm_output_lanes_ring<64,64>", "k_wino_gemm_output_lanes_ring<32,32>",
                                      "k_wino_gemm_output_lanes_ring<32,64>"};   // channels, tiles of a workgroup
  plan.name = names[form];
  return plan_set(plan, f.kernel, dim3(8 * a.ny * a.slots), dim3(64 * f.waves), lds, a, ArgBlock{}, ArgOut{a.out}, ArgBias{});
}

}  // namespace ehip
