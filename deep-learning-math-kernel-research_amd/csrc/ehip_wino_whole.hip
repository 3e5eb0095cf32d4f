// Planning of the kernel that runs a Winograd layer whole (ehip_wino_whole.hpp).  No kernels here.
#include "ehip_internal.hpp"

namespace ehip {

struct WholeSplit {
  int waves;               // of a workgroup
  int splits, per_split;   // workgroups of a block of tiles, groups of 16 output channels of each
};
static WholeSplit whole_split(int nks, int blocks, int groups)
{
  // eight waves where no CU gets a second block (128 -> 128, 196 blocks: 17.8 against 22.1 us), else four, so that the phases of two
  // or three blocks overlap on a CU (402 blocks: 29.6 against 31.9; 64 -> 64, 784 blocks: 28.0 against 41.6)
  WholeSplit s;
  s.waves = blocks <= 256 || nks > 2 ? 8 : 4;
  if (const char *env = getenv("EHIP_WINO_WHOLE_WAVES")) s.waves = env[0] == '8' || nks > 2 ? 8 : 4;
  // fewer blocks than CUs: the output channels of a block are shared out, as long as that leaves every wave some
  s.splits = 256 / blocks;
  const int most = (groups + s.waves - 1) / s.waves;
  s.splits = s.splits > most ? most : s.splits;
  if (const char *env = getenv("EHIP_WINO_WHOLE_SPLITS")) s.splits = atoi(env);
  s.splits = s.splits < 1 ? 1 : s.splits > groups ? groups : s.splits;
  s.per_split = (groups + s.splits - 1) / s.splits;
  s.splits = (groups + s.per_split - 1) / s.per_split;
  return s;
}

// Where one kernel is the faster one.  It saves a launch, the trip of the transformed input through memory and the start of a second
// kernel with cold caches; it pays with input transforms that the workgroups sharing a block of tiles repeat, with weights
// that every block streams for itself, and with phases that overlap only where a CU holds several workgroups.  So it wins
// while the blocks of 16 tiles come to about one round of workgroups, for longer the fewer channels there are, and from more
// blocks on the more input channels a workgroup transforms for itself; from fewer with at most 64 output channels, because
// half of the waves then stay out of the weights' way.  u8 in / s8 out, time of this kernel over that of the stages at so many
// blocks of tiles, other tensors on every call, some 300 MB in turn (the same ones again and again are kinder to it, 0.70
// for 128 -> 128 at 196 blocks, but a model does not repeat its layers):
//   tile size 6: 64 -> 64, 4 / 40 / 98 / 245 / 392 / 784 blocks 0.99 / 0.92 / 0.89 / 0.72 / 0.83 / 0.91 (and slower between ResNet-50's other
//     layers); 64 -> 128, 40 / 98 / 392 / 784 0.99 / 0.93 / 0.92 / 1.04; 64 -> 256, 245 / 392 0.93 / 1.12; 128 -> 48, 40 / 64 / 245 / 469 1.04 / 0.97 / 0.69 / 0.74;
//     128 -> 128, 64 / 98 / 160 / 469 1.13 / 0.98 / 0.81 / 0.83; 128 -> 256, 98 / 160 / 245 0.86 / 1.02 / 0.94; 192 -> 64, 64 / 98 / 129 1.01 / 0.93 / 0.81;
//     192 -> 128, 98 / 129 1.15 / 0.82; 192 -> 256, 129 / 196 0.99 / 0.97; 256 -> 64, 98 / 129 0.96 / 0.85; 256 -> 128, 98 / 129 / 196 1.19 / 0.89 / 0.78; 256 -> 256,
//     129 / 196 1.15 / 1.05
//   tile size 5: 64 -> 64, 5 / 244 / 790 0.93 / 0.72 / 0.87; 64 -> 128, 16 / 41 / 384 0.99 / 0.94 / 0.85; 64 -> 256, 244 / 384 0.88 / 1.05; 128 -> 48, 16 / 41 0.98 / 0.93;
//     128 -> 128, 65 / 100 / 469 1.04 / 0.92 / 0.82; 128 -> 256, 244 / 394 0.92 / 0.95; 192 -> 64, 65 0.94; 192 -> 128, 100 / 125 1.03 / 0.88; 192 -> 256, 163 / 244
//     0.97 / 0.94; 256 -> 64, 65 0.83; 256 -> 128, 100 / 125 1.07 / 0.88; 256 -> 256, 163 1.02
//   tile size 4: 64 -> 128, 4 / 784 0.84 / 0.93; 64 -> 256, 392 / 784 0.86 / 1.02; 128 -> 128, 40 / 65 / 466 0.97 / 0.95 / 0.82; 128 -> 256, 392 0.94; 128 -> 512, 160 1.12;
//     192 -> 64, 65 0.91; 192 -> 128, 98 / 123 1.03 / 0.92; 192 -> 256, 160 / 245 0.98 / 0.91; 256 -> 128, 98 / 123 1.03 / 0.91; 256 -> 256, 196 / 245 0.95 / 0.98
// and where the stages have the kernel that shares the columns of the positions out (ehip_wino_cols.hip), planes of 14 x 14 / 12 x 12 / 8 x 8:
//   tile size 6: 64 -> 64, 64 / 98 / 196 blocks 1.09 / 0.92 / 0.82; 64 -> 128, 32 / 48 / 98 1.16 / 1.02 / 0.96; 128 -> 64, 64 / 98 / 128 1.31 / 1.03 / 0.90; 128 -> 128, 64 / 98 / 128
//     1.33 / 1.03 / 0.95; 192 -> 64, 64 / 98 1.40 / 0.98; 256 -> 64, 64 / 98 / 128 1.30 / 1.04 / 0.98
//   tile size 5: 64 -> 64, 16 / 64 / 98 1.03 / 1.00 / 0.90; 64 -> 128, 32 / 48 1.11 / 0.96; 128 -> 64, 64 / 98 1.16 / 0.96; 128 -> 128, 64 / 98 1.21 / 0.99; 192 -> 64, 98 / 128
//     1.08 / 0.94; 256 -> 64, 98 / 128 1.00 / 0.94
//   tile size 4: 128 -> 128, 64 / 98 1.12 / 0.95; 256 -> 64, 64 / 98 1.09 / 0.99
// A wave takes whole groups of 16 output channels, so 9 groups cost four waves as much as 12 and eight as much as 16.  Where the waves go
// through more than one round of them it pays (`full`) with eight waves from so many CUs on whose waves would all be at work, 2000 random
// layers:
//   tile size 6: 64 -> 160, 133 / 144 / 157 blocks (82 / 89 / 108 CUs) 1.19 / 1.15 / 1.09; 64 -> 144, 192 / 196 / 224 / 256 (108 / 110 / 126 / 144) 1.08 / 0.94 / 0.93 / 0.94; 64 ->
//     176, 179 (123) 0.90; 192 -> 160, 172 (107) 1.11; 192 -> 144, 204 / 222 (115 / 125) 0.92 / 0.93
//   tile size 5: 64 -> 160 .. 256, 135 to 256 (110 to 224) 1.01 to 0.89; 128 -> 144 .. 192, 144 to 188 (81 to 118) 1.13 to 1.06, 252 (205) 0.90; 192 -> 144 /
//     160, 179 / 167 (101 / 104) 1.18 / 1.16
//   tile size 4, by blocks: up to 128 channels 0.77 to 0.98; 192, 154 to 160 1.04, 180 / 196 0.90; 256 -> 160 .. 208, 153 / 160 1.08 / 0.97
// with four waves, tile size 6 only next to the next round of blocks (two rounds of groups, 260 / 300 / 341 / 378 blocks 1.35 / 1.24 / 1.11 / 1.11); tile
//   size 5, two rounds, 257 to 319 blocks 1.19 to 1.04, 324 to 522 0.97 to 0.87, three, 258 to 384 1.16 to 1.06, 387 to 398 0.95; tile size 4, three or
//   four, 128 channels, 259 to 338 blocks 1.11 to 1.05, 359 to 392 0.96 to 0.93, 64 channels 0.82 to 0.92.
// (Points on either side of a line differ by 2 to 5 %, about what two boxes differ by: nearer than that a line is not known.)
static bool wino_whole_pays(int A, int nks, int blocks, int groups)
{
  // blocks from (at most 64 output channels; more) and to, groups of 16 output channels, blocks x groups; by k-steps of 64 input
  // channels
  struct Limit { int least_few, least, most, groups, work, full; };
  static const Limit limits[3][4] = {
      {{1, 1, 1200, 64, 6300, 0}, {1, 90, 480, 16, 6300, 0}, {56, 110, 256, 16, 4000, 165}, {90, 115, 256, 12, 3200, 160}},     // tile size 4
      {{1, 40, 1200, 64, 4700, 112}, {80, 90, 480, 16, 4000, 120}, {110, 110, 256, 16, 4000, 120}, {110, 120, 256, 8, 4000, 120}},
      {{24, 56, 400, 64, 3300, 109}, {110, 112, 480, 8, 4000, 109}, {95, 128, 256, 12, 4000, 109}, {110, 128, 256, 8, 4000, 109}}};
  // (the fused stage with a workgroup of its own on a CU for every 16 channels x 16 tiles: the stages)
  if (A >= 5 && (long long)blocks * groups <= 256) return false;
  const Limit &l = limits[A - 4][nks - 1];
  if (blocks < (groups <= 4 ? l.least_few : l.least) || blocks > l.most || groups > l.groups || (long long)blocks * groups > l.work) return false;
  const WholeSplit s = whole_split(nks, blocks, groups);
  const int rounds = (s.per_split + s.waves - 1) / s.waves;   // of a wave's groups of output channels
  if (rounds == 1) return true;
  if (s.waves == 8) return A == 4 ? blocks >= l.full : blocks * groups >= l.full * 8 * rounds;
  if (A == 6) return blocks >= 384 && blocks * 4 * rounds <= l.work;
  return A == 5 ? blocks >= (rounds == 2 ? 320 : 385) : rounds == 2 || nks == 1 || blocks >= 350;
}

bool wino_whole_applies(const WinoArgs &w, const WinoFusedArgs &f)
{
  const int nks = (f.ic2 + 3) / 4;
  // what the kernel can run: u8 codes, the transformed input of sixteen tiles in LDS (up to 256 input channels), input and packed
  // weights addressed with 32 bits, f32 output without the in-place sum
  const unsigned long long bytes = (unsigned long long)w.n * w.ic2 * w.ih * w.iw * 16;
  const unsigned long long weights = (unsigned long long)f.tile * f.tile * f.units_pad * f.ocpp * 16;
  if (nks > 4 || !w.in_u8 || f.units_pad < 4 * nks || bytes > 0xffffff00ull || weights > 0x7fffffffull ||
      (f.out_type == EHIP_F32 && f.with_sum))
    return false;
  const char *env = getenv("EHIP_WINO_WHOLE");
  if (env && env[0] == '0') return false;
  if (env && env[0] == '1') return true;
  // (a switch that asks for a form of the separate stages asks for the stages)
  for (const char *k : {"EHIP_WINO_LANES", "EHIP_WINO_LANES_WRES", "EHIP_WINO_LANES_SLOTS", "EHIP_WINO_LANES_WAVES", "EHIP_WINO_RING",
                        "EHIP_WINO_COLS", "EHIP_WINO_BUF_GATHER", "EHIP_WINO_WIDE_GATHER", "EHIP_WINO_SHORT"})
    if (getenv(k)) return false;
  return wino_whole_pays(f.tile, nks, (f.t + 15) / 16, f.oc2);
}

hipError_t plan_wino_whole(LaunchPlan &plan, const WinoArgs &w, const WinoFusedArgs &f)
{
  WinoWholeArgs a;
  memset(&a, 0, sizeof(a));
  a.w = w;
  a.f = f;
  const int nks = (f.ic2 + 3) / 4;
  a.nx = (f.t + 15) / 16;
  const WholeSplit split = whole_split(nks, a.nx, f.oc2);
  const WholeForm form = f.tile == 4 ? wino_whole_form4(nks, split.waves, f.out_type, f.with_sum != 0)
      : f.tile == 5 ? wino_whole_form5(nks, split.waves, f.out_type, f.with_sum != 0) : wino_whole_form6(nks, split.waves, f.out_type, f.with_sum != 0);
  a.splits = split.splits;
  a.per_split = split.per_split;
  a.nt_magic = div_magic(f.nt);
  a.wt_magic = div_magic(f.wt);
  plan.name = "k_wino_whole";
  return plan_set(plan, form.kernel, dim3((unsigned)((long long)a.nx * a.splits + 7) / 8 * 8), dim3(64 * form.waves), form.lds, a, ArgBlock{}, ArgIn{nullptr}, ArgOut{nullptr}, ArgBias{});
}

}  // namespace ehip
